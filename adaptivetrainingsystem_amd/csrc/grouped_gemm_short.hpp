// Grouped bfloat16 NT products with a short K per group: the weight gradients of experts that got a few hundred rows
// (included by grouped_gemm.hip).
//
// Such a product mostly writes: 8 gradients of [28672, 4096] over 128 rows each read 70 MB and write 1.9 GB.  The 256 x 256
// tile of the long products holds a CU alone, and with two slabs of K its set-up, first loads and epilogue follow one
// another with nothing beside them: 10 us for 128 KB, 3.3 TB/s.  Here a workgroup is four waves with a 128 x 128 tile and
// one 32 KB slab of LDS, so that four of them share a CU and the loads of one run beside the stores of another, and the
// results leave with non-temporal stores (nobody reads them before the last-level cache has been overwritten several times;
// with plain ones 588 -> 529 us in the first row below).  Slabs, swizzle, MFMA shape and order over K are those of
// grouped_gemm_dma16_kernel: the same bits.  Rows per expert, 256 x 256 tiles -> this, microseconds (stores alone at 5.7 TB/s):
//   8 x [28672, 4096]  (330)   100: 586 -> 420   190: 680 -> 554   320: 907 -> 752   450: 1056 -> 965   600: 1246 (1265)
//   8 x [4096, 14336]  (165)   100: 324 -> 210   190: 371 -> 270   320: 475 -> 374   450:  556 -> 475   600:  642 -> 582
//   64 x [2816, 2048]  (130)   100: 256 -> 176   190: 322 -> 231   320: 383 -> 303   450:  455 (454)    600:  507 (558)
//   64 x [2048, 1408]   (65)   100: 162 ->  91   190: 207 -> 122   320: 229 -> 152   450:  276 -> 205   600:  290 (305)
// With 128 x 256 tiles, two workgroups per CU, the first row reads 433, 580, 780, 991.
#pragma once

namespace ats {

constexpr int kShortBM = 128, kShortBN = 128;

__global__ __launch_bounds__(256, 4) void grouped_gemm_short_kernel(GroupedArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef bf16_t T;
    constexpr int BM = kShortBM, BN = kShortBN, NW = 4, TM = 4, TN = 4;
    constexpr int NI = BM / 8 / NW;                       // load instructions per wave and operand: 8 rows of 128 bytes each
    __shared__ __align__(16) unsigned char smem[(BM + BN) * 128];
    typedef __attribute__((address_space(3))) void* lds_ptr_t;

    TileCoord tc;
    if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc)) return;
    const int count = p.row_count[tc.e];
    const int row0 = p.row_start[tc.e];
    const int nk = (p.k_count ? p.k_count[tc.e] : p.K) / 64;
    const int tile_row = tc.mt * BM;
    const T* A = static_cast<const T*>(p.a_ptrs ? p.a_ptrs[tc.e] : p.a) + ((p.a_ptrs ? 0 : row0) + (int64_t)tile_row) * p.lda;
    const T* B = static_cast<const T*>(p.b[tc.e]) + (int64_t)tc.nt * BN * p.ldb;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    constexpr int kRsrcFlags = 0x00020000;
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(A), 0, -1, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(B), 0, -1, kRsrcFlags);
    const int drow = lane >> 3, dchunk = (lane & 7) ^ drow;
    unsigned ao[NI], bo[NI];
#pragma unroll
    for (int j = 0; j < NI; ++j) {      // rows past the end of the group or of N repeat the last one (never stored)
        const int r = (j * NW + wave) * 8 + drow;
        const int m = tile_row + r < count ? r : count - 1 - tile_row;
        const int n = tc.nt * BN + r < p.N_out ? r : p.N_out - 1 - tc.nt * BN;
        ao[j] = (unsigned)((int64_t)m * p.lda * 2 + dchunk * 16);
        bo[j] = (unsigned)((int64_t)n * p.ldb * 2 + dchunk * 16);
    }
    unsigned char* const dma = smem + wave * 1024;
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int frow = lane & 15, kgrp = lane >> 4;
    for (int kt = 0; kt < nk; ++kt) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_ptr_t)(dma + j * NW * 1024), 16, ao[j], kt * 128, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_ptr_t)(dma + BM * 128 + j * NW * 1024), 16, bo[j], kt * 128, 0, 0);
        }
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int slot = ((4 * ks + kgrp) ^ (frow & 7)) * 16;
            const unsigned char* fa = smem + (wm * 64 + frow) * 128 + slot;
            const unsigned char* fb = smem + BM * 128 + (wn * 64 + frow) * 128 + slot;
            union {
                u32x4_t u;
                bf16x8_t v;
            } a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i].u = *reinterpret_cast<const u32x4_t*>(fa + i * 2048);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j].u = *reinterpret_cast<const u32x4_t*>(fb + j * 2048);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j].v, a[i].v, acc[j][i], 0, 0, 0);
        }
        // every wave has read its fragments: the slab (or the epilogue's staging) may be overwritten
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    typedef AccView16<TM, TN, false> View;
    constexpr int WSTAGE = epilogue_wstage_bytes<T, View, false>();
    static_assert(NW * WSTAGE <= (BM + BN) * 128, "epilogue staging exceeds the slab");
    epilogue_view<T, View, false, false, false, true>(View{acc}, smem + wave * WSTAGE, static_cast<T*>(p.out), p.ldo,
                                  (int64_t)row0 + tile_row + wm * 64, count - tile_row - wm * 64, tc.nt * BN + wn * 64, p.N_out,
                                  lane);
#endif
}

static int launch_short(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + kShortBN - 1) / kShortBN;
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = max_rows / (p.E > 0 ? p.E : 1) >= kAlignedBandsMinAvgRows ? 1 : 0;
    const int64_t blocks = grid_blocks(max_rows, p.E, kShortBM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(grouped_gemm_short_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p);
    return ATS_OK;
}

}  // namespace ats
