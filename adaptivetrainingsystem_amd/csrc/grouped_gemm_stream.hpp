// Grouped NT products of groups with a few rows: the launch is a stream of weights (included by grouped_gemm.hip).
//
// What bounds it is the order in which the memory sees the weights.  A stand-alone reader of a [28672, 4096] bfloat16
// matrix whose workgroups walk panels of R rows, C bytes of each row per step, reads at 5.6-6.2 TB/s with R x C = 128 x
// 128 bytes (the shape of a wide tile's slabs), 4.3-5.6 with 32 x 512, and 6.5-7.0 with 16 x 1024 and longer pieces of
// fewer rows (non-temporal loads, two or more steps in flight).  So a workgroup owns 16 weight rows (32 with NP = 2; with
// the SwiGLU epilogue 16 gate rows and the matching 16 up rows) over all of K and its four waves split K in 256-byte
// pieces: together they read 1 KB of each of the rows per step, two steps ahead.  A wave's piece goes through registers
// into wave-private LDS (coalesced in, MFMA fragments out, no barrier: a wave's LDS accesses complete in order); at the
// end the waves' float32 accumulators are added in wave order.  Activations (up to 16 MT rows per group and tile) come
// from L2 the same way; rows that a group does not have are not read.
#pragma once

namespace ats {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float acc16_t;
template <typename T>
__device__ __forceinline__ void mma16_step(const u32x4_t& wfrag, const u32x4_t& afrag, acc16_t& c);
template <>
__device__ __forceinline__ void mma16_step<bf16_t>(const u32x4_t& wfrag, const u32x4_t& afrag, acc16_t& c) {
    union {
        u32x4_t u;
        bf16x8_t v;
    } w, a;
    w.u = wfrag;
    a.u = afrag;
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.v, a.v, c, 0, 0, 0);
}
template <>
__device__ __forceinline__ void mma16_step<float>(const u32x4_t& wfrag, const u32x4_t& afrag, acc16_t& c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wfrag.x), __uint_as_float(afrag.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wfrag.y), __uint_as_float(afrag.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wfrag.z), __uint_as_float(afrag.z), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wfrag.w), __uint_as_float(afrag.w), c, 0, 0, 0);
}

template <int NP, int MT, int KW>
struct StreamTile {
    static constexpr int kRows = 16 * MT, kWRows = 16 * NP;   // activation and weight rows of a tile
    static constexpr int kPitch = 256 + 16;
    static constexpr int kStage = (16 + kWRows) * kPitch;     // bytes per wave: the weight rows, 16 activation rows
    static constexpr int kRedPitch = kWRows + 4;
    static constexpr int kLds = KW * (kStage > kRows * kRedPitch * 4 ? kStage : kRows * kRedPitch * 4);
};

// Block -> (group, m-tile, n-tile).  The panels of all groups form one list (a group's n-tiles in turn, its m-tiles innermost), dealt to
// the XCDs (block % 8) in whole rounds of `chunk` panels each, what is left (chunk 0: everything) in eight equal pieces, so that no XCD
// has more than its share: in supertiles of 32, the order of the wide tiles, 17 experts of 64 panels are 34 supertiles, five on some XCDs
// and four on others.  One piece per XCD is the fastest for many small groups, an XCD then reads a few weights at a time: 64 experts
// [2816, 2048] + [2048, 1408], whole layer, 24 tokens 183.5 us in supertiles, 181 in chunks, 179 in pieces; 128 experts of 768, 60 tokens
// 309 -> 281 -> 279.  Eight large experts, one to an XCD, would be slower than in chunks (64 tokens 457 against 469), and sixteen with
// skewed routing (41 tokens of 16 x [11264, 2048] 113 -> 109 in chunks, 118 in pieces): pieces from 32 experts on.
__device__ __forceinline__ bool decode_panel_wave(unsigned block, const int32_t* __restrict__ row_count, int E, int BM, int n_tiles,
                                                  unsigned chunk, TileCoord* out) {
    const int lane = threadIdx.x & 63;
    int t0 = 0, p0 = 0;
    unsigned total = 0;
    for (int g0 = 0; g0 < E; g0 += 64) {
        int t, p;
        tile_scan64(row_count, E, E, g0, BM, 1, false, lane, &t, &p);
        if (g0 == 0) t0 = t, p0 = p;
        total += (unsigned)__builtin_amdgcn_readlane(p, 63);
    }
    const unsigned all = total * (unsigned)n_tiles, xcd = block % kNumXcd, li = block / kNumXcd;
    const unsigned whole = chunk ? all / (kNumXcd * chunk) * chunk : 0;      // an XCD's panels in whole rounds
    if (li < whole) block = (li / chunk * kNumXcd + xcd) * chunk + li % chunk;
    else {
        const unsigned rest = all - kNumXcd * whole, per = (rest + kNumXcd - 1) / kNumXcd, at = xcd * per + li - whole;
        if (li - whole >= per || at >= rest) return false;
        block = kNumXcd * whole + at;
    }
    const int pos = (int)(block / (unsigned)n_tiles);      // in the list of all groups' m-tiles
    int base = 0;
    for (int g0 = 0; g0 < E; g0 += 64) {
        int t = t0, p = p0;
        if (g0 > 0) tile_scan64(row_count, E, E, g0, BM, 1, false, lane, &t, &p);
        const unsigned long long hit = __ballot(base + p > pos);
        if (hit) {
            const int first = __ffsll((long long)hit) - 1;
            const unsigned tiles = (unsigned)__builtin_amdgcn_readlane(t, first);
            const unsigned at = block - (unsigned)(base + __builtin_amdgcn_readlane(p, first) - (int)tiles) * (unsigned)n_tiles;
            out->e = g0 + first;
            out->nt = (int)(at / tiles);
            out->mt = (int)(at % tiles);
            return true;
        }
        base += __builtin_amdgcn_readlane(p, 63);
    }
    return false;
}

template <typename T, typename TO, int NP, int MT, int KW, bool SWIGLU>
__global__ __launch_bounds__(KW * 64, KW == 4 && MT <= 2 ? 3 : 2) void grouped_gemm_stream_kernel(GroupedArgs p) {
    typedef StreamTile<NP, MT, KW> Tile;
    constexpr int PITCH = Tile::kPitch;
    constexpr int VEC = 16 / (int)sizeof(T);
    constexpr int BK = 256 / (int)sizeof(T);
    constexpr int NIW = 4 * NP, NIX = 4 * MT;                 // load instructions per piece: 4 rows x 256 bytes each
    constexpr int kCols = SWIGLU ? Tile::kWRows / 2 : Tile::kWRows;   // output columns of a tile
    static_assert(!SWIGLU || NP == 2, "the SwiGLU tile is a panel of gate rows and one of up rows");

    extern __shared__ __align__(16) unsigned char smem[];

    TileCoord tc;
    if (!decode_panel_wave(blockIdx.x, p.row_count, p.E, Tile::kRows, p.n_tiles, (unsigned)p.sm, &tc)) return;
    const int count = p.row_count[tc.e];
    const int row0 = p.row_start[tc.e];
    const int K = p.K;
    const T* Bexp = static_cast<const T*>(p.b[tc.e]);
    const T* A = static_cast<const T*>(p.a_ptrs ? p.a_ptrs[tc.e] : p.a);
    const int arow0 = p.a_ptrs ? 0 : row0;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane >> 4, lchunk = lane & 15;
    const int m0 = tc.mt * Tile::kRows;
    const int n0 = min(tc.nt * kCols, p.N_out - kCols);       // the last tile of a ragged N repeats columns of the one before
    const int rows = __builtin_amdgcn_readfirstlane(min(count - m0, Tile::kRows));

    // instruction i reads 4 weight rows: a uniform base and one offset per lane
    const T* wbase[NIW];
#pragma unroll
    for (int i = 0; i < NIW; ++i)
        wbase[i] = Bexp + (int64_t)(SWIGLU && i >= 4 ? p.up_offset + n0 + (i - 4) * 4 : n0 + i * 4) * p.ldb;
    const unsigned woff = (unsigned)(lrow * (int)p.ldb + lchunk * VEC);
    const T* xp[NIX];
#pragma unroll
    for (int i = 0; i < NIX; ++i) {
        int m = m0 + i * 4 + lrow;
        m = m < count ? m : count - 1;
        int64_t src = arow0 + m;
        if (p.a_rows) src = p.a_rows[src] / p.a_row_div;
        xp[i] = A + src * p.lda + lchunk * VEC;
    }

    acc16_t acc[NP][MT];
#pragma unroll
    for (int j = 0; j < NP; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = acc16_t{0.f, 0.f, 0.f, 0.f};

    const int nk = (K + BK - 1) / BK;
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};
    unsigned char* const stage = smem + wave * Tile::kStage;
    unsigned char* const st_at = stage + lrow * PITCH + lchunk * 16;
    const unsigned char* const fr_at = stage + (lane & 15) * PITCH + (lane >> 4) * 16;
    // the fragments of the last 16 activation rows cover rows that do not exist: zeros
#pragma unroll
    for (int i = 0; i < NIX; ++i)
        if (i * 4 >= rows) xp[i] = nullptr;

    u32x4_t w[2][NIW], x[NIX];
    auto load_w = [&](int piece, u32x4_t(&rw)[NIW]) {
        if (piece >= nk) return;                              // wave-uniform
        const unsigned koff = (unsigned)piece * BK;
        const bool ok = (int)koff + lchunk * VEC < K;         // false only in the last piece of a ragged K
#pragma unroll
        for (int i = 0; i < NIW; ++i)
            rw[i] = ok ? __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wbase[i] + (woff + koff))) : zero4;
    };
    auto load_x = [&](int piece, int i16) {                   // 16 activation rows
        const int koff = piece * BK;
        const bool ok = piece < nk && koff + lchunk * VEC < K;
#pragma unroll
        for (int i = 4 * i16; i < 4 * i16 + 4; ++i)
            x[i] = ok && xp[i] ? *reinterpret_cast<const u32x4_t*>(xp[i] + koff) : zero4;
    };
    auto step = [&](int piece, u32x4_t(&rw)[NIW]) {
        if (piece >= nk) return;
#pragma unroll
        for (int i = 0; i < NIW; ++i) *reinterpret_cast<u32x4_t*>(st_at + i * 4 * PITCH) = rw[i];
        load_w(piece + 2 * KW, rw);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (i > 0 && i * 16 >= rows) continue;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<u32x4_t*>(st_at + (Tile::kWRows + q * 4) * PITCH) = x[4 * i + q];
            load_x(piece + KW, i);
            // other lanes' pieces are read below (the wave's LDS accesses themselves are in order)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const u32x4_t fx = *reinterpret_cast<const u32x4_t*>(fr_at + Tile::kWRows * PITCH + ks * 64);
#pragma unroll
                for (int j = 0; j < NP; ++j)
                    mma16_step<T>(*reinterpret_cast<const u32x4_t*>(fr_at + j * 16 * PITCH + ks * 64), fx, acc[j][i]);
            }
            asm volatile("" ::: "memory");                    // the next rows' writes stay behind these reads
        }
    };
    load_w(wave, w[0]);
#pragma unroll
    for (int i = 0; i < MT; ++i)
        if (i == 0 || i * 16 < rows) load_x(wave, i);
    load_w(wave + KW, w[1]);
    for (int s = wave; s < nk; s += 2 * KW) {
        step(s, w[0]);
        step(s + KW, w[1]);
    }

    // ---- add the waves' partial tiles in wave order
    __syncthreads();
    float* const red = reinterpret_cast<float*>(smem);
    {
        float* mine = red + (wave * Tile::kRows + (lane & 15)) * Tile::kRedPitch + 4 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < NP; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
                *reinterpret_cast<float4*>(mine + i * 16 * Tile::kRedPitch + j * 16) =
                    make_float4(acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]);
    }
    __syncthreads();
    constexpr int GROUPS = kCols / 4;
    TO* out = static_cast<TO*>(p.out);
    for (int t = tid; t < rows * GROUPS; t += KW * 64) {
        const int r = t / GROUPS, c = t % GROUPS * 4;
        if (n0 + c >= p.N_out) continue;
        auto sum = [&](int col) {
            float4 v = *reinterpret_cast<const float4*>(red + r * Tile::kRedPitch + col);
#pragma unroll
            for (int q = 1; q < KW; ++q) {
                const float4 u = *reinterpret_cast<const float4*>(red + (q * Tile::kRows + r) * Tile::kRedPitch + col);
                v.x += u.x;
                v.y += u.y;
                v.z += u.z;
                v.w += u.w;
            }
            return v;
        };
        float4 v = sum(c);
        if constexpr (SWIGLU) {
            const float4 u = sum(16 + c);
            v.x = silu_f(v.x) * u.x;
            v.y = silu_f(v.y) * u.y;
            v.z = silu_f(v.z) * u.z;
            v.w = silu_f(v.w) * u.w;
        }
        TO* dst = out + ((int64_t)row0 + m0 + r) * p.ldo + n0 + c;
        if constexpr (sizeof(TO) == 4) *reinterpret_cast<float4*>(dst) = v;
        else *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
    }
}

template <typename T, typename TO, int NP, int MT, int KW, bool SWIGLU>
static int launch_stream(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    typedef StreamTile<NP, MT, KW> Tile;
    constexpr int kCols = SWIGLU ? Tile::kWRows / 2 : Tile::kWRows;
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + kCols - 1) / kCols;
    p.sm = p.E >= 32 ? 0 : 32;      // panels of a chunk
    auto kern = grouped_gemm_stream_kernel<T, TO, NP, MT, KW, SWIGLU>;
    if (Tile::kLds > 64 * 1024) {
        static LdsReservation reserved;
        hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern)}, Tile::kLds);
        if (e != hipSuccess) {
            set_error("grouped GEMM: cannot reserve %d bytes of LDS: %s", Tile::kLds, hipGetErrorString(e));
            return ATS_ERR_LAUNCH;
        }
    }
    // a tile has at least one row; a multiple of 8, so that every XCD has room for an eighth
    const int64_t blocks = (std::min(max_rows, max_rows / Tile::kRows + p.E) * p.n_tiles + kNumXcd - 1) / kNumXcd * kNumXcd;
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(KW * 64), Tile::kLds, s, p);
    return ATS_OK;
}

}  // namespace ats
