// Grouped bfloat16 NT products of groups with some dozens of rows, and products of one group with up to a few hundred: the weights are
// most of what is read, and each is used by up to 128 rows (included by grouped_gemm.hip).
//
// What bounds it is again the stream of weights.  A workgroup is four waves with a tile of up to 128 activation rows x 128 weight rows,
// a wave 32 of these against all of the activations.  Both operands go straight to LDS in slabs of 64 elements, weights two slabs ahead
// (and activations of up to 64 rows; taller slabs one, a third stage of them would not leave room for a second workgroup on the CU, whose
// loads run beside this one's barriers, first loads and epilogue).  Experts' weights that no other tile reads are loaded non-temporally:
// 64 groups of 24 rows, gate/up [2816, 2048] 131 -> 119 us, 8 x [28672, 4096] 325 -> 294.  (A single weight is not: a linear layer that is
// called again soon finds part of it in the last-level cache, 32 decoding steps of 64 sequences of 2048 4.13 -> 3.96 ms.)  And no two neighbouring tiles walk K in step: with rows
// of 4, 8 or 28 KB the same columns of all rows lie in a few of the memory's channels, so tile nt of a group starts at slab 5 nt and
// comes round to it (one group, whose workgroups already hold different slices or fit the caches, starts at 0):
//   8 x [28672, 4096], 64 rows each 388 -> 323 us, 100 rows 393 -> 344;  8 x [4096, 14336], 24 rows 182 -> 138 (6.8 TB/s), 64 rows 183 -> 155
//   64 x [2816, 2048], 64 rows 162 -> 132, 100 rows 177 -> 143
// Against the kernels that took these sizes before (32- and 64-row tiles with K split in the workgroup, register-staged 128-row tiles,
// the 256-row tile, weight streams, slices of K with their sum), microseconds, weights from HBM:
//   rows per group              16          24          48          64          96
//   64 x gate/up [2816, 2048]   122 -> 115  158 -> 118  162 -> 122  163 -> 132  176 -> 143
//   64 x [2048, 1408]            65 ->  59   72 ->  60   77 ->  66   80 ->  71   87 ->  78
//   8 x gate/up [28672, 4096]   287 -> 279  353 -> 282  365 -> 300  366 -> 325  377 -> 329
//   8 x [4096, 14336]           156 -> 137  166 -> 138  175 -> 149  177 -> 154  183 -> 168
//   one group, rows             40          64          128         200         300         512
//   [6144, 4096]                 22 ->  18   25 ->  20   32 ->  27   50 ->  34   59 ->  34   62 ->  47
//   [4096, 4096]                 17 ->  16   19 ->  18   24 ->  21   33 ->  27   59 ->  34   63 ->  36
//   [2048, 2048]                                                     18 ->  15   29 ->  17   31 ->  18    (1000 rows 33 -> 20)
// Sums over K are sequential in float32 from the tile's first slab on; with one group that is the order of grouped_gemm_dma16_kernel.
#pragma once

namespace ats {

constexpr int kBandRows = 128, kBandCols = 128;     // most activation rows and weight rows of a tile
constexpr int kBandWStage = kBandCols * 128;        // bytes of a slab of weights: 64 elements of every row
constexpr int kBandLds = 80 * 1024;                 // two workgroups per CU

// MT: 16-row fragments of activations.  once: weights to be loaded non-temporally.  k0: first slab.
template <typename TO, bool SWIGLU, int MT>
__device__ __forceinline__ void band_tile(const GroupedArgs& p, unsigned char* smem, const bf16_t* A, const bf16_t* Bexp, int nt, int row0,
                                          int count, int tile_row, int nk, bool once, int k0, TO* out) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef bf16_t T;
    constexpr int NW = 4, HALF = kBandCols / 2;
    constexpr int NIA = MT / 2, NIB = kBandCols / 8 / NW;       // load instructions per wave and slab: 8 rows of 128 bytes each
    constexpr int AS = MT * 16 * 128;                           // bytes of a slab of activations
    constexpr int AR = MT <= 4 ? 3 : 2;                         // stages of its ring
    constexpr int A_BASE = 3 * kBandWStage;
    static_assert(A_BASE + AR * AS <= kBandLds, "LDS of the rings");
    typedef __attribute__((address_space(3))) void* lds_ptr_t;

    const int arow0 = p.a_ptrs ? 0 : row0;
    const bool gather = p.a_rows != nullptr;
    const T* a_base = gather ? A : A + ((int64_t)arow0 + tile_row) * p.lda;
    constexpr int kRsrcFlags = 0x00020000;                      // raw buffer, 32-bit data format
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a_base), 0, (int)p.a_extent_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(Bexp), 0, (int)p.b_extent_bytes, kRsrcFlags);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int drow = lane >> 3, dchunk = (lane & 7) ^ drow;
    // rows past the end of the group repeat its last one (never stored); without a gather the loads are of some word and not used
    const int32_t* const index = gather ? p.a_rows + arow0 : p.row_count;
    int a_idx[NIA];
#pragma unroll
    for (int j = 0; j < NIA; ++j) {
        const int m = tile_row + (j * NW + wave) * 8 + drow;
        a_idx[j] = index[gather ? (m < count ? m : count - 1) : 0];
    }
    unsigned ao[NIA], bo[NIB];
#pragma unroll
    for (int j = 0; j < NIB; ++j) {      // as do columns past the end of N
        const int r = (j * NW + wave) * 8 + drow;
        int n, up = 0;
        if (SWIGLU) {
            n = nt * HALF + (r & (HALF - 1));
            up = r >= HALF ? p.up_offset : 0;
        } else n = nt * kBandCols + r;
        n = (n < p.N_out ? n : p.N_out - 1) + up;
        bo[j] = (unsigned)((int64_t)n * p.ldb * 2 + dchunk * 16);
    }
    unsigned char* const dma_b = smem + wave * 1024;
    unsigned char* const dma_a = smem + A_BASE + wave * 1024;
    auto issue_b = [&](int kt, int stage) {
        kt = kt + k0 < nk ? kt + k0 : kt + k0 - nk;
        if (once) {
#pragma unroll
            for (int j = 0; j < NIB; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(dma_b + stage + j * NW * 1024), 16, bo[j], kt * 128, 0, kNonTemporal);
        } else {
#pragma unroll
            for (int j = 0; j < NIB; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(dma_b + stage + j * NW * 1024), 16, bo[j], kt * 128, 0, 0);
        }
    };
    auto issue_a = [&](int kt, int stage) {
        kt = kt + k0 < nk ? kt + k0 : kt + k0 - nk;
#pragma unroll
        for (int j = 0; j < NIA; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(dma_a + stage + j * NW * 1024), 16, ao[j], kt * 128, 0, 0);
    };
    issue_b(0, 0);
    if (nk > 1) issue_b(1, kBandWStage);
#pragma unroll
    for (int j = 0; j < NIA; ++j) asm volatile("" : "+v"(a_idx[j]));      // the indices are waited for behind the weights' first loads
#pragma unroll
    for (int j = 0; j < NIA; ++j) {
        const int r = (j * NW + wave) * 8 + drow, last = count - 1 - tile_row;
        const int src = gather ? a_idx[j] / p.a_row_div : (r < last ? r : last);
        ao[j] = (unsigned)((int64_t)src * p.lda * 2 + dchunk * 16);
    }
    issue_a(0, 0);
    if (AR == 3 && nk > 1) issue_a(1, AS);

    f32x4_t acc[2][MT];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int frow = lane & 15, kgrp = lane >> 4;
    const unsigned char* fa_addr[2];
    const unsigned char* fb_addr[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int slot = ((4 * ks + kgrp) ^ (frow & 7)) * 16;
        fa_addr[ks] = smem + A_BASE + frow * 128 + slot;
        fb_addr[ks] = smem + (wave * (SWIGLU ? 16 : 32) + frow) * 128 + slot;
    }
    int sb = 0, sa = 0;                  // stages of slab kt
    for (int kt = 0; kt < nk; ++kt) {
        // the youngest loads are the weights (and, with three stages, the activations) of the slab after this one
        if (kt + 1 == nk) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else if (kt == 0) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AR == 3 ? NIA : 0) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AR == 3 ? NIA + NIB : NIB) : "memory");
        const int sb2 = sb == 0 ? 2 * kBandWStage : sb - kBandWStage;             // stage of slab kt + 2
        if (AR == 3) {
            if (kt + 2 < nk) issue_a(kt + 2, sa == 0 ? 2 * AS : sa - AS);
        } else if (kt + 1 < nk) issue_a(kt + 1, AS - sa);
        if (kt + 2 < nk) issue_b(kt + 2, sb2);
        union Frag {
            u32x4_t u;
            bf16x8_t v;
        };
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            Frag w[2], a[MT];
#pragma unroll
            for (int j = 0; j < 2; ++j) w[j].u = *reinterpret_cast<const u32x4_t*>(fb_addr[ks] + sb + j * (SWIGLU ? HALF : 16) * 128);
#pragma unroll
            for (int i = 0; i < MT; ++i) a[i].u = *reinterpret_cast<const u32x4_t*>(fa_addr[ks] + sa + i * 2048);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j].v, a[i].v, acc[j][i], 0, 0, 0);
        }
        sb = sb == 2 * kBandWStage ? 0 : sb + kBandWStage;
        sa = AR == 3 ? (sa == 2 * AS ? 0 : sa + AS) : AS - sa;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");               // the slabs give way to the epilogue's staging
    typedef AccView16<MT, 2, SWIGLU> View;
    constexpr int WSTAGE = epilogue_wstage_bytes<TO, View, false>();
    static_assert(NW * WSTAGE <= kBandLds, "epilogue staging exceeds the rings");
    epilogue_view<TO, View, SWIGLU>(View{acc}, smem + wave * WSTAGE, out, p.ldo, (int64_t)row0 + tile_row, count - tile_row,
                                    SWIGLU ? nt * HALF + wave * 16 : nt * kBandCols + wave * 32, p.N_out, lane);
#endif
}

template <typename TO, bool SWIGLU, bool SLICED>
__global__ __launch_bounds__(256, 2) void grouped_gemm_band_kernel(GroupedArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    TileCoord tc;
    if (!decode_panel_wave(blockIdx.x, p.row_count, p.E, p.tile_rows, SLICED ? p.n_tiles * p.k_splits : p.n_tiles, (unsigned)p.sm, &tc)) return;
    const int e = __builtin_amdgcn_readfirstlane(tc.e), mt = __builtin_amdgcn_readfirstlane(tc.mt);
    int nt = __builtin_amdgcn_readfirstlane(tc.nt), K = p.K;
    const int count = __builtin_amdgcn_readfirstlane(p.row_count[e]), row0 = __builtin_amdgcn_readfirstlane(p.row_start[e]);
    const bf16_t* B = static_cast<const bf16_t*>(p.b[e]);
    const bf16_t* A = static_cast<const bf16_t*>(p.a_ptrs ? p.a_ptrs[e] : p.a);
    TO* out = static_cast<TO*>(p.out);
    if constexpr (SLICED) {
        const int split = nt / p.n_tiles;
        nt -= split * p.n_tiles;
        A += (int64_t)split * p.k_slice;
        B += (int64_t)split * p.k_slice;
        out += split * p.part_stride;
        K = p.k_slice;
    }
    // a group's tiles have one height, in pairs of fragments
    const int m_tiles = (count + p.tile_rows - 1) / p.tile_rows;
    const int height = ((count + m_tiles - 1) / m_tiles + 31) / 32 * 32;
    const int tile_row = mt * height;
    if (tile_row >= count) return;
    const bool experts = p.E > 1, once = experts && m_tiles == 1;
    const int nk = K / 64, k0 = experts ? 5 * nt % nk : 0;
    switch (height) {
        case 32: return band_tile<TO, SWIGLU, 2>(p, smem, A, B, nt, row0, count, tile_row, nk, once, k0, out);
        case 64: return band_tile<TO, SWIGLU, 4>(p, smem, A, B, nt, row0, count, tile_row, nk, once, k0, out);
        case 96: return band_tile<TO, SWIGLU, 6>(p, smem, A, B, nt, row0, count, tile_row, nk, once, k0, out);
        default: return band_tile<TO, SWIGLU, 8>(p, smem, A, B, nt, row0, count, tile_row, nk, once, k0, out);
    }
}

template <typename TO, bool SWIGLU, bool SLICED>
static int launch_band(const GroupedArgs& p0, int64_t max_rows, int tile_rows, hipStream_t s) {
    GroupedArgs p = p0;
    constexpr int kCols = SWIGLU ? kBandCols / 2 : kBandCols;
    p.n_tiles = (p.N_out + kCols - 1) / kCols;
    // panels of a chunk (see decode_panel_wave).  Down projections in chunks: 64 unequal groups of 48 rows on average 84 -> 73 us, 8 x
    // [4096, 14336] in two slices 156 -> 138; gate/up in eight pieces: 8 groups of 24 rows 298 -> 286.
    p.sm = SWIGLU ? 0 : 16;
    p.tile_rows = tile_rows;
    auto kern = grouped_gemm_band_kernel<TO, SWIGLU, SLICED>;
    static LdsReservation reserved;
    hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern)}, kBandLds);
    if (e != hipSuccess) {
        set_error("grouped GEMM: cannot reserve %d bytes of LDS: %s", kBandLds, hipGetErrorString(e));
        return ATS_ERR_LAUNCH;
    }
    const int64_t tiles = std::min(max_rows, max_rows / tile_rows + p.E) * p.n_tiles * (SLICED ? p.k_splits : 1);
    const int64_t blocks = (tiles + kNumXcd - 1) / kNumXcd * kNumXcd;
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), kBandLds, s, p);
    return ATS_OK;
}

}  // namespace ats
