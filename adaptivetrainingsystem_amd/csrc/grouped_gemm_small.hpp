// Grouped NT products whose grid of large tiles would leave most of the chip idle (included by grouped_gemm.hip).
//
// A [512, 512] x [512, 512]^T product is four 256 x 256 tiles: four workgroups on 256 CUs, each walking all of K.
// Here a wave owns a 32 TM x 32 TN tile (64 x 64 or 32 x 32), and a workgroup is
//   KW = 4:           one such tile, whose four waves split K between them: wave w takes the 128-byte slabs w, w + 4,
//                     ... of the reduction, so that a tile is four times shorter and the chip sees 16-64 times as
//                     many workgroups; at the end the waves' float32 accumulators are added in LDS in wave order;
//   KW = 1, WG = 2:   2 x 2 such tiles, each over all of K in the order of the large float32 tiles (the same bits).
// Every wave works alone until the end: its slab goes through registers into a wave-private piece of LDS (coalesced
// 128-byte row pieces in, MFMA fragments out; a wave's LDS accesses complete in order, so there is no barrier in the
// loop) while the next slab is in flight.  Results leave through LDS as 16-byte (8-byte for bfloat16) stores.  No
// atomics: the result does not depend on timing.  Any K that is a multiple of 16 bytes.
//
// BKM (float32): the weights are stored [K][N], the reduction index along their rows, as the data gradient of a linear layer
// finds them; AKM: the other operand too, [K][rows] (the weight gradient: tokens along the rows of both, the rows of the
// second one optionally gathered).  A slab is then 32 rows of K, staged as it lies, and a lane's four reduction steps are four
// 4-byte reads instead of one of 16: the same values in the same order as from a transposed copy, without the copy.  In AKM
// every group has p.uniform_rows output rows, so no table is read.  512 rows
// x [512, 1024] with the copy 41 -> 11 us.
#pragma once

namespace ats {

template <typename T, typename TO, int TM, int TN, int KW, int WG, bool SWIGLU>
struct SmallTile {
    static constexpr int BM = 32 * TM, BN = 32 * TN;                      // of a wave
    static constexpr int kWaves = KW * WG * WG;
    static constexpr int kCols = SWIGLU ? BN / 2 : BN;                    // output columns of a wave's tile
    static constexpr int kRows = BM * WG, kTileCols = kCols * WG;         // output of a workgroup
    static constexpr int kStage = (BM + BN) * kRowPitch;                  // bytes per wave
    static constexpr int kRedPitch = BN + 4;                              // floats per row of a wave's tile
    static constexpr int kRed = BM * kRedPitch * 4;                       // bytes per wave
    static constexpr int kLds = kWaves * (kStage > kRed ? kStage : kRed);
};

template <typename T, typename TO, int TM, int TN, int KW, int WG, bool SWIGLU, bool AKM = false, bool BKM = false>
__global__ __launch_bounds__(KW* WG* WG * 64) void grouped_gemm_small_kernel(GroupedArgs p) {
    typedef SmallTile<T, TO, TM, TN, KW, WG, SWIGLU> Tile;
    constexpr int BM = Tile::BM, BN = Tile::BN;
    constexpr int VEC = 16 / (int)sizeof(T);
    constexpr int BK = 128 / (int)sizeof(T);
    constexpr int NIA = BM / 8, NIB = BN / 8;   // load instructions per slab: 8 rows x 128 bytes each
    constexpr int HALF = BN / 2;
    static_assert(!SWIGLU || TN % 2 == 0, "SwiGLU needs gate and up tiles in the same wave");

    extern __shared__ __align__(16) unsigned char smem[];

    static_assert(!AKM || BKM, "K-major rows come with K-major weights");
    static_assert(!BKM || (sizeof(T) == 4 && !SWIGLU), "K-major operands: the plain float32 product");
    TileCoord tc;
    if constexpr (AKM) {
        const int per = (p.uniform_rows + Tile::kRows - 1) / Tile::kRows * p.n_tiles;
        tc.e = blockIdx.x / per;
        tc.mt = blockIdx.x % per / p.n_tiles;
        tc.nt = blockIdx.x % per % p.n_tiles;
    } else {
        if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, Tile::kRows, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc)) return;
    }
    const int count = AKM ? p.uniform_rows : p.row_count[tc.e];
    const int64_t row0 = AKM ? (int64_t)tc.e * count : p.row_start[tc.e];
    const int K = p.k_count ? p.k_count[tc.e] : p.K;
    const int k_row0 = AKM && p.k_start ? p.k_start[tc.e] : 0;
    const T* Bexp = AKM ? reinterpret_cast<const T*>(p.b) : static_cast<const T*>(p.b[tc.e]);
    const T* A = static_cast<const T*>(p.a_ptrs ? p.a_ptrs[tc.e] : p.a);
    const int64_t arow0 = p.a_ptrs ? 0 : row0;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave % KW;                                   // slice of K
    const int m0 = tc.mt * Tile::kRows + wave / KW / WG * BM;   // the wave's first row and output column
    const int n0 = tc.nt * Tile::kTileCols + wave / KW % WG * Tile::kCols;
    const int lrow = lane >> 3, lchunk = lane & 7;

    // rows past the end of the group or of N repeat the last one (their results are never stored)
    const T* ap[NIA];
#pragma unroll
    for (int i = 0; i < NIA && !AKM; ++i) {
        int m = m0 + i * 8 + lrow;
        m = m < count ? m : count - 1;
        int64_t src = arow0 + m;
        if (p.a_rows) src = p.a_rows[src] / p.a_row_div;
        ap[i] = A + src * p.lda + lchunk * VEC;
    }
    const T* bp[NIB];
    // K-major: lanes per row of a slab, rows per load instruction; columns past the end repeat the last four (never stored)
    constexpr int CA = BM / 4, RA = 64 / CA, PA = BM * 4 + 16, CB = BN / 4, RB = 64 / CB, PB = BN * 4 + 16;
    const T* const akm = A + min(m0 + lane % CA * 4, count - 4);
    const T* const bkm = Bexp + min(n0 + lane % CB * 4, p.N_out - 4);
#pragma unroll
    for (int i = 0; i < NIB && !BKM; ++i) {
        const int rb = i * 8 + lrow;
        int n = n0 + (SWIGLU && rb >= HALF ? rb - HALF : rb);
        n = n < p.N_out ? n : p.N_out - 1;
        const int brow = SWIGLU && rb >= HALF ? p.up_offset + n : n;
        bp[i] = Bexp + (int64_t)brow * p.ldb + lchunk * VEC;
    }

    f32x16_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;

    const int nk = (K + BK - 1) / BK;
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};
    u32x4_t ra[NIA], rb[NIB];
    unsigned char* const stage = smem + wave * Tile::kStage;
    unsigned char* const st_at = stage + lrow * kRowPitch + lchunk * 16;
    const unsigned char* const fr_at = stage + (lane & 31) * kRowPitch + (lane >> 5) * 16;

    // K-major: rows past K repeat the last one and are cleared on their way into LDS, so that no load has a branch of its own;
    // the gathered rows' numbers are asked for a slab ahead of the rows
    int rn[NIB];
    auto rows_of = [&](int slab) {
#pragma unroll
        for (int i = 0; i < NIB; ++i) rn[i] = p.b_rows[k_row0 + min(slab * BK + i * RB + lane / CB, K - 1)];
    };
    const bool gathered = AKM && p.b_rows;
    auto load = [&](int slab) {
        const int koff = slab * BK;
        const bool ok = koff + lchunk * VEC < K;    // false only in the last slab of a ragged K
#pragma unroll
        for (int i = 0; i < NIA; ++i) {
            if constexpr (AKM) {
                const int k = min(koff + i * RA + lane / CA, K - 1);
                ra[i] = *reinterpret_cast<const u32x4_t*>(akm + ((int64_t)k_row0 + k) * p.lda);
            } else ra[i] = ok ? *reinterpret_cast<const u32x4_t*>(ap[i] + koff) : zero4;
        }
#pragma unroll
        for (int i = 0; i < NIB; ++i) {
            if constexpr (BKM) {
                const int64_t r = gathered ? rn[i] / p.b_row_div : (int64_t)k_row0 + min(koff + i * RB + lane / CB, K - 1);
                rb[i] = *reinterpret_cast<const u32x4_t*>(bkm + r * p.ldb);
            } else rb[i] = ok ? *reinterpret_cast<const u32x4_t*>(bp[i] + koff) : zero4;
        }
    };
    // four reduction steps of a lane from a slab as it lies
    auto column = [&](const unsigned char* at, int pitch, int ks) {
        u32x4_t f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            f[c] = *reinterpret_cast<const uint32_t*>(at + (8 * ks + 4 * (lane >> 5) + c) * pitch + (lane & 31) * 4);
        return f;
    };
    if (kw < nk) {
        if (gathered) rows_of(kw);
        load(kw);
        if (gathered && kw + KW < nk) rows_of(kw + KW);
    }
    for (int s = kw; s < nk; s += KW) {
        if (BKM && (s + 1) * BK > K) {
#pragma unroll
            for (int i = 0; i < NIA; ++i)
                if (AKM && s * BK + i * RA + lane / CA >= K) ra[i] = zero4;
#pragma unroll
            for (int i = 0; i < NIB; ++i)
                if (s * BK + i * RB + lane / CB >= K) rb[i] = zero4;
        }
#pragma unroll
        for (int i = 0; i < NIA; ++i)
            *reinterpret_cast<u32x4_t*>(AKM ? stage + (i * RA + lane / CA) * PA + lane % CA * 16 : st_at + i * 8 * kRowPitch) = ra[i];
#pragma unroll
        for (int i = 0; i < NIB; ++i)
            *reinterpret_cast<u32x4_t*>(BKM ? stage + BM * kRowPitch + (i * RB + lane / CB) * PB + lane % CB * 16
                                            : st_at + (BM + i * 8) * kRowPitch) = rb[i];
        // other lanes' pieces are read below: nothing may move across (the wave's LDS accesses themselves are in order)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (s + KW < nk) {
            load(s + KW);
            if (gathered && s + 2 * KW < nk) rows_of(s + 2 * KW);
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4_t fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                fa[i] = AKM ? column(stage + i * 128, PA, ks)
                            : *reinterpret_cast<const u32x4_t*>(fr_at + i * 32 * kRowPitch + ks * 32);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[j] = BKM ? column(stage + BM * kRowPitch + j * 128, PB, ks)
                            : *reinterpret_cast<const u32x4_t*>(fr_at + (BM + j * 32) * kRowPitch + ks * 32);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) mma_step<T>(fb[j], fa[i], acc[j][i]);
        }
        asm volatile("" ::: "memory");   // the next slab's writes stay behind these reads
    }

    // ---- through LDS; the partial tiles of the K slices are added in their order
    __syncthreads();
    float* const red = reinterpret_cast<float*>(smem);
    {
        float* mine = red + wave * (BM * Tile::kRedPitch) + (lane & 31) * Tile::kRedPitch + 4 * (lane >> 5);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(mine + i * 32 * Tile::kRedPitch + j * 32 + 8 * q) =
                        make_float4(acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
    }
    __syncthreads();
    constexpr int GROUPS = Tile::kCols / 4;      // groups of 4 output columns per row of a wave's tile
    TO* out = static_cast<TO*>(p.out);
    constexpr int PER_TILE = BM * GROUPS;
    for (int t = tid; t < WG * WG * PER_TILE; t += Tile::kWaves * 64) {
        const int tile = t / PER_TILE, r = t % PER_TILE / GROUPS, c = t % GROUPS * 4;
        const int m = tc.mt * Tile::kRows + tile / WG * BM + r;
        const int n = tc.nt * Tile::kTileCols + tile % WG * Tile::kCols + c;
        if (m >= count || n >= p.N_out) continue;
        const float* part = red + (tile * KW * BM + r) * Tile::kRedPitch;
        auto sum = [&](int col) {
            float4 v = *reinterpret_cast<const float4*>(part + col);
#pragma unroll
            for (int w = 1; w < KW; ++w) {
                const float4 u = *reinterpret_cast<const float4*>(part + w * BM * Tile::kRedPitch + col);
                v.x += u.x;
                v.y += u.y;
                v.z += u.z;
                v.w += u.w;
            }
            return v;
        };
        float4 v = sum(c);
        if constexpr (SWIGLU) {
            const float4 u = sum(HALF + c);
            v.x = silu_f(v.x) * u.x;
            v.y = silu_f(v.y) * u.y;
            v.z = silu_f(v.z) * u.z;
            v.w = silu_f(v.w) * u.w;
        }
        TO* dst = out + ((int64_t)row0 + m) * p.ldo + n;
        if constexpr (sizeof(TO) == 4) *reinterpret_cast<float4*>(dst) = v;
        else *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
    }
}

template <typename T, typename TO, int TM, int TN, int KW, int WG, bool SWIGLU, bool AKM = false, bool BKM = false>
static int launch_small(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    typedef SmallTile<T, TO, TM, TN, KW, WG, SWIGLU> Tile;
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + Tile::kTileCols - 1) / Tile::kTileCols;
    static_assert(!BKM || 32 * (Tile::BN * 4 + 16) <= Tile::BN * kRowPitch, "a slab as it lies fits the room of its rows");
    auto kern = grouped_gemm_small_kernel<T, TO, TM, TN, KW, WG, SWIGLU, AKM, BKM>;
    if (Tile::kLds > 64 * 1024) {
        static LdsReservation reserved;
        hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern)}, Tile::kLds);
        if (e != hipSuccess) {
            set_error("grouped GEMM: cannot reserve %d bytes of LDS: %s", Tile::kLds, hipGetErrorString(e));
            return ATS_ERR_LAUNCH;
        }
    }
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = 0;
    const int64_t blocks = AKM ? (int64_t)p.E * ((p.uniform_rows + Tile::kRows - 1) / Tile::kRows) * p.n_tiles
                               : grid_blocks(max_rows, p.E, Tile::kRows, p.n_tiles, p.sm, p.sn, false);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(Tile::kWaves * 64), Tile::kLds, s, p);
    return ATS_OK;
}

}  // namespace ats
