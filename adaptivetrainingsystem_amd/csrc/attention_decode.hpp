// Attention of a few query rows against a long cache (included by attention.hip): one new position per sequence, all
// query heads of a kv head together, at most 16 rows.  The call is one pass over K and V, so what counts is how the
// memory sees it: a workgroup's four waves take the 32-key chunks of its (batch, kv head) in turn, each wave for itself
// with its own running maximum, sum and output, so that a chunk of K and one of V (8 KB each, contiguous) are in flight
// per wave while the previous ones are worked on, and no barrier ever holds a wave back.  The wide kernel this replaces at
// these sizes keeps the four waves in step over 64-key tiles, of which three only help to load.  Measured (32 / 8 heads,
// D 128, one new token): 64 sequences x 2048 keys 91 -> 82 us (6.5 TB/s), x 4096 189 -> 161 (6.7), 8 x 2048 27 -> 16.
//
// S^T = K . Q^T and O^T = V^T . P^T on 16 x 16 x 32 MFMAs: the accumulators of S^T (lane: row l % 16, keys 4 g + c of two
// 16-key tiles, g = l / 16) are the B operand of the second product in the key order {4 g + c, 16 + 4 g + c}, and V^T
// is read in the same order through two transposing LDS reads per fragment.  K and V pass through one wave-private LDS
// region one after the other.
#pragma once

namespace ats {

constexpr int kDecRows = 16;     // query rows of a workgroup (positions x heads of the kv group)
constexpr int kDecKeys = 32;     // keys of a wave's chunk
constexpr int kDecWaves = 4;
template <int D>
constexpr int decode_lds_bytes() {
    constexpr int stage = kDecKeys * (D * 2 + 32), merge = kDecRows * (D + 4) * 4;
    return kDecWaves * (stage > merge ? stage : merge) + kDecWaves * kDecRows * 8;
}

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float dec_acc_t;
__device__ __forceinline__ dec_acc_t dec_mma(const au32x4_t& a, const au32x4_t& b, dec_acc_t c) {
    union {
        au32x4_t u;
        abf16x8_t v;
    } x, y;
    x.u = a;
    y.u = b;
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, y.v, c, 0, 0, 0);
}
// with the lanes 16 and 32 positions away (all 64 lanes active)
__device__ __forceinline__ float groups_max(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return xor32_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
__device__ __forceinline__ float groups_sum(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return xor32_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// part_out == nullptr: the workgroup sees all keys and writes out / lse; otherwise part p of n_parts sees part_len keys
// from p * part_len (the last part the rest) and leaves its rows for attention_merge_kernel.
template <int D, bool BIAS>
__global__ __launch_bounds__(kDecWaves * 64, 3) void attention_decode_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, int64_t k_sb, int64_t k_sh, const bf16_t* __restrict__ v,
    int64_t v_sb, int v_sl, int64_t v_sh, const float* __restrict__ key_bias, bf16_t* __restrict__ out,
    float* __restrict__ lse, float* __restrict__ part_out, int Hq, int Hkv, int L, int Lk, float scale_log2, int n_groups,
    int n_parts, int part_len) {
    constexpr int LPR = D / 8;                    // lanes per row of K or V, 16 bytes each
    constexpr int RPI = 64 / LPR;                 // rows per load instruction
    constexpr int NL = kDecKeys / RPI;            // load instructions per chunk
    constexpr int KS = D / 32, DB = D / 16;
    constexpr int KPITCH = D * 2 + 16, VPITCH = D * 2 + 32;
    constexpr int STAGE = kDecKeys * VPITCH;
    extern __shared__ __align__(16) unsigned char smem[];

    const int part = blockIdx.x / n_groups, group = blockIdx.x - part * n_groups;
    const int b = group / Hkv, hkv = group - b * Hkv;
    const int rep = Hq / Hkv, n_rows = L * rep;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, g = lane >> 4;

    const int row = col < n_rows ? col : n_rows - 1;            // rows past the last repeat it and are not stored
    const int pos = row / rep;
    const bf16_t* qp = q + ((int64_t)(b * Hq + hkv * rep + row - pos * rep) * L + pos) * D;
    au32x4_t qf[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const au32x4_t*>(qp + s * 32 + g * 8);
    const int last_key = pos + Lk - L;                          // last key that this lane's row sees

    const int k_first = part * part_len;
    const int k_end = part == n_parts - 1 ? Lk : k_first + part_len;
    const int n_chunks = (k_end - k_first + kDecKeys - 1) / kDecKeys;
    const float* bias_row = BIAS ? key_bias + (int64_t)b * Lk : nullptr;

    // keys past the last of the cache read as zeros
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(k + b * k_sb + hkv * k_sh), 0, (int)((int64_t)Lk * D * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(v + b * v_sb + hkv * v_sh), 0, (int)((((int64_t)Lk - 1) * v_sl + D) * 2), 0x00020000);
    const int lrow = lane / LPR, lchunk = lane % LPR;
    unsigned char* const stage = smem + wave * STAGE;
    au32x4_t rk[NL], rv[NL];
    constexpr int kNt = 2;                                      // non-temporal: every byte is read once
    auto load_k = [&](int chunk) {
        const int base = (k_first + chunk * kDecKeys) * D * 2;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            rk[i] = __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, ((i * RPI + lrow) * D + lchunk * 8) * 2, base, kNt);
    };
    auto load_v = [&](int chunk) {
        const int base = (k_first + chunk * kDecKeys) * v_sl * 2;
#pragma unroll
        for (int i = 0; i < NL; ++i)
            rv[i] = __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, ((i * RPI + lrow) * v_sl + lchunk * 8) * 2, base, kNt);
    };

    dec_acc_t acc_o[DB];
#pragma unroll
    for (int d = 0; d < DB; ++d) acc_o[d] = dec_acc_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    if (wave < n_chunks) {
        load_k(wave);
        load_v(wave);
    }
    // one row and one chunk column per lane, 16 bytes; fragments: K rows by lane l % 16, V through transposing reads
    unsigned char* const k_st = stage + lrow * KPITCH + lchunk * 16;
    unsigned char* const v_st = stage + lrow * VPITCH + lchunk * 16;
    const unsigned char* const k_fr = stage + col * KPITCH + g * 16;
    const unsigned char* const v_fr = stage + (4 * g + (col >> 2)) * VPITCH + (col & 3) * 8;
    for (int c = wave; c < n_chunks; c += kDecWaves) {
        const int key0 = k_first + c * kDecKeys;
        const bool more = c + kDecWaves < n_chunks;
        // ---- scores
#pragma unroll
        for (int i = 0; i < NL; ++i) *reinterpret_cast<au32x4_t*>(k_st + i * RPI * KPITCH) = rk[i];
        if (more) load_k(c + kDecWaves);
        // other lanes' pieces are read below (a wave's LDS accesses themselves are in order)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        dec_acc_t s[2] = {dec_acc_t{0.f, 0.f, 0.f, 0.f}, dec_acc_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                s[t] = dec_mma(*reinterpret_cast<const au32x4_t*>(k_fr + t * 16 * KPITCH + ks * 64), qf[ks], s[t]);
        asm volatile("" ::: "memory");
        // ---- V into the same region; its fragments are read behind the softmax
#pragma unroll
        for (int i = 0; i < NL; ++i) *reinterpret_cast<au32x4_t*>(v_st + i * RPI * VPITCH) = rv[i];
        if (more) load_v(c + kDecWaves);
        // ---- softmax: this lane's 8 keys of its row
        float sv[8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                float val = s[t][x] * scale_log2;
                if constexpr (BIAS) {
                    const int key = key0 + t * 16 + 4 * g + x;
                    val += (key < Lk ? bias_row[key] : 0.f) * 1.4426950408889634f;
                }
                sv[t * 4 + x] = val;
            }
        if (key0 + kDecKeys - 1 > Lk - L || key0 + kDecKeys > k_end) {      // some key is past a row's last or the part's end
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int key = key0 + t * 16 + 4 * g + x;
                    if (key > last_key || key >= k_end) sv[t * 4 + x] = -INFINITY;
                }
        }
        float mx = sv[0];
#pragma unroll
        for (int x = 1; x < 8; ++x) mx = fmaxf(mx, sv[x]);
        mx = groups_max(mx);
        // the reference point follows the maximum only when that has grown by more than 8 (log2 units), see attention_q_tile
        const float m_new = mx - m_run > 8.0f ? mx : m_run;          // (-inf) - (-inf) is not greater: stays -inf
        const float m_use = m_new == -INFINITY ? 0.f : m_new;         // no visible key yet: all p are 0
        if (!__all(m_new == m_run)) {
            const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_use);
            l_run *= alpha;
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
                for (int x = 0; x < 4; ++x) acc_o[d][x] *= alpha;
            m_run = m_new;
        }
        float p[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            p[x] = __builtin_amdgcn_exp2f(sv[x] - m_use);
            l_run += p[x];
        }
        const au32x4_t pf = {pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]), pack_bf16x2(p[4], p[5]), pack_bf16x2(p[6], p[7])};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int d = 0; d < DB; ++d) {
            union {
                att_tr_t t[2];
                au32x4_t u;
            } f;
            f.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((att_lds_tr_ptr_t)(v_fr + d * 32));
            f.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((att_lds_tr_ptr_t)(v_fr + d * 32 + 16 * VPITCH));
            acc_o[d] = dec_mma(f.u, pf, acc_o[d]);
        }
        asm volatile("" ::: "memory");
    }
    l_run = groups_sum(l_run);

    // ---- merge the waves: out = sum_w 2^(m_w - M) O_w / sum_w 2^(m_w - M) l_w
    __syncthreads();
    constexpr int OPITCH = D + 4;
    float* const so = reinterpret_cast<float*>(smem);
    float* const sml = reinterpret_cast<float*>(smem + decode_lds_bytes<D>() - kDecWaves * kDecRows * 8);
    {
        float* mine = so + (wave * kDecRows + col) * OPITCH + 4 * g;
#pragma unroll
        for (int d = 0; d < DB; ++d)
            *reinterpret_cast<float4*>(mine + d * 16) = make_float4(acc_o[d][0], acc_o[d][1], acc_o[d][2], acc_o[d][3]);
        if (g == 0) *reinterpret_cast<float2*>(sml + (wave * kDecRows + col) * 2) = make_float2(m_run, l_run);
    }
    __syncthreads();
    const int r = tid >> 4, c8 = (tid & 15) * (D / 16);
    if (r >= n_rows) return;
    float M = -INFINITY, w[kDecWaves], l = 0.f;
#pragma unroll
    for (int i = 0; i < kDecWaves; ++i) M = fmaxf(M, sml[(i * kDecRows + r) * 2]);
#pragma unroll
    for (int i = 0; i < kDecWaves; ++i) {
        const float m = sml[(i * kDecRows + r) * 2];
        w[i] = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
        l += w[i] * sml[(i * kDecRows + r) * 2 + 1];
    }
    float o[D / 16];
#pragma unroll
    for (int j = 0; j < D / 16; j += 4) {
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < kDecWaves; ++i) {
            const float4 u = *reinterpret_cast<const float4*>(so + (i * kDecRows + r) * OPITCH + c8 + j);
            a.x += w[i] * u.x;
            a.y += w[i] * u.y;
            a.z += w[i] * u.z;
            a.w += w[i] * u.w;
        }
        o[j] = a.x;
        o[j + 1] = a.y;
        o[j + 2] = a.z;
        o[j + 3] = a.w;
    }
    const int rpos = r / rep, hq = hkv * rep + r - rpos * rep;
    if (part_out) {
        float* dst = part_out + (((int64_t)(b * Hq + hq) * L + rpos) * n_parts + part) * (D + kPartPad);
#pragma unroll
        for (int j = 0; j < D / 16; j += 4)
            *reinterpret_cast<float4*>(dst + c8 + j) = make_float4(o[j], o[j + 1], o[j + 2], o[j + 3]);
        if ((tid & 15) == 0) *reinterpret_cast<float2*>(dst + D) = make_float2(M, l);
        return;
    }
    const float inv = 1.0f / l;
    bf16_t* orow = out + ((int64_t)b * L + rpos) * (int64_t)(Hq * D) + hq * D + c8;
#pragma unroll
    for (int j = 0; j < D / 16; j += 4)
        *reinterpret_cast<uint2*>(orow + j) =
            make_uint2(pack_bf16x2(o[j] * inv, o[j + 1] * inv), pack_bf16x2(o[j + 2] * inv, o[j + 3] * inv));
    if (lse && (tid & 15) == 0) lse[(int64_t)(b * Hq + hq) * L + rpos] = (M + log2f(l)) * 0.6931471805599453f;
}

}  // namespace ats
