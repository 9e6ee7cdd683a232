// Grouped expert GEMMs for gfx950 (CDNA4 MFMA, wave64).
//
//   gate/up + SwiGLU : h[r, i] = silu(a_r . Wgu[e][i,:]) * (a_r . Wgu[e][I+i,:])
//   down             : y[r, :] = h[r,:] . Wd[e]^T
//
// Both are "NT" products: activations [rows, K] and weights [N, K] have K contiguous, so both operands are
// fetched with 16-byte loads along K and fed to the matrix cores without any transpose.  The weight fragment
// is the first MFMA operand, so the accumulator of a lane holds 4 consecutive output columns of one output
// row.  With SwiGLU a tile holds BN/2 gate rows and the matching BN/2 up rows, so silu(g)*u is formed in
// registers and the [rows, 2I] intermediate never exists.  The permutation gather is fused into the A load
// (row index table).  One launch covers all experts: tile_schedule.hpp maps a block id to (expert, m-tile,
// n-tile) so that the 32 workgroups of an XCD share operand panels in that XCD's L2.
//
// Kernels, by the rows per expert the host sees (launch_grouped):
//   grouped_gemm_dma16_kernel     bf16, groups above 192 rows and large launches (prefill and fine-grained shapes; also the
//                                 training instances that save g/u or apply the SwiGLU gradient).  256 x 256
//                                 tile, 8 waves of 128 x 64 on v_mfma_f32_16x16x32_bf16, K in 64-element
//                                 slabs that go from memory straight into LDS (buffer_load ... lds: unpadded
//                                 128-byte rows, XOR swizzle on the global side), three activation stages and
//                                 two weight stages in the 160 KiB of LDS, one barrier per slab, fragment
//                                 reads and loads placed among the MFMAs with sched_group_barrier.
//   grouped_gemm_dma_kernel       the same data path for float32 operands on v_mfma_f32_32x32x2_f32.
//   grouped_gemm_pipelined_kernel register-staged, two padded stages (144-byte pitch): the 128-row tiles of mid-sized
//                                 groups, the 32 / 64-row tiles that cut K into slices over workgroups, and gather
//                                 sources whose lane offsets do not fit 32 bits.
//   grouped_gemm_stream_kernel    decode-sized groups: a stream of weights, see grouped_gemm_stream.hpp.
//   grouped_gemm_small_kernel     32 and 64-row tiles for launches whose large tiles would leave most CUs idle, see
//                                 grouped_gemm_small.hpp.
//   grouped_gemm_short_kernel     weight gradients over a few hundred rows per expert: stores bound, see
//                                 grouped_gemm_short.hpp.
//   grouped_gemm_kernel           general fallback for K that is not a multiple of a slab (bounds-checked loads).
#include <math.h>

#include <type_traits>

#include "ats_common.hpp"
#include "tile_schedule.hpp"

namespace ats {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
// Native 16-byte vector (plain IR loads/stores, so staging arrays stay in registers).
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

struct GroupedArgs {
    const void* a;           // [*, K] activations
    const void* const* a_ptrs;  // optional: per expert A base; its rows are then counted from 0 (no row_start)
    const int32_t* a_rows;   // optional gather table over the row space
    int a_row_div;
    int64_t lda;             // elements
    const void* const* b;    // per expert weight [N_total, K]
    int64_t ldb;             // elements between rows of b
    const int32_t* k_count;  // optional: per expert K (a multiple of the K slab), overrides K
    void* out;               // [*, N_out]
    int64_t ldo;
    const int32_t* row_start;
    const int32_t* row_count;
    int E, K, N_out, up_offset, n_tiles;
    int sm, sn;              // supertile shape of the launch (sm * sn = 32 blocks), see tile_schedule.hpp
    int aligned_bands;       // 1: every group's tile count is rounded up to a multiple of sm
    // split K (register-staged kernel only): k_splits > 1 turns every expert into k_splits groups that each
    // multiply a K / k_splits wide slice and write a partial result part_stride elements apart
    int k_splits, k_slice;   // k_slice = K / k_splits
    int64_t part_stride;
    // direct-to-LDS path only: bytes addressable from the A / B descriptors (0 = path not usable)
    uint32_t a_extent_bytes, b_extent_bytes;
    // training (direct-to-LDS kernel only): the gate / up pre-activations, [*, 2 * N_out]; written by the
    // forward instance, read by the instance whose epilogue turns dh into the gradients of g and u
    void* gu_out;
    int64_t ld_gu;
    // training, bf16 instances of the direct-to-LDS kernel, optional: the tile's result also goes, transposed,
    // into t_out[column, t_col0[group] + row inside the group] (row stride ld_t elements), zero in the columns
    // between a group's last row and the next multiple of 64: the layout that the weight-gradient product
    // contracts over (see ats_wgrad_plan), so that no transposing pass over the activations is needed
    void* t_out;
    int64_t ld_t;
    const int32_t* t_col0;
    int tile_rows;          // MIDROWS instance: most rows of a tile (0: the tile's own height)
    // float32 products with both operands K-major: output rows of every group, first row of K per group (null: 0), optional
    // gather of the second operand's rows; p.b is that operand itself
    int uniform_rows, b_row_div;
    const int32_t* k_start;
    const int32_t* b_rows;
};

constexpr int kNonTemporal = 2;  // cache policy of a buffer load
constexpr int kRowPitch = 144;  // bytes per staged row: 128 data + 16 pad

template <typename T>
__device__ __forceinline__ void mma_step(const u32x4_t& wfrag, const u32x4_t& afrag, f32x16_t& c);

template <>
__device__ __forceinline__ void mma_step<bf16_t>(const u32x4_t& wfrag, const u32x4_t& afrag, f32x16_t& c) {
    union {
        u32x4_t u;
        bf16x8_t v;
    } w, a;
    w.u = wfrag;
    a.u = afrag;
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w.v, a.v, c, 0, 0, 0);
}
template <>
__device__ __forceinline__ void mma_step<float>(const u32x4_t& wfrag, const u32x4_t& afrag, f32x16_t& c) {
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(wfrag.x), __uint_as_float(afrag.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(wfrag.y), __uint_as_float(afrag.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(wfrag.z), __uint_as_float(afrag.z), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(wfrag.w), __uint_as_float(afrag.w), c, 0, 0, 0);
}

}  // namespace ats

#include "grouped_gemm_small.hpp"
#include "grouped_gemm_stream.hpp"

namespace ats {

// Views of a wave's accumulators, 32 output rows at a time, as groups of 4 consecutive output columns
// per lane.  ib: 32-row block of the wave's sub-tile, g: group, half: 0 = gate (or the plain product),
// 1 = the matching up column.  All indices are compile-time constants after unrolling.
// 32 x 32 x 16 MFMA: lane holds row (lane & 31), columns 8 q + 4 (lane >> 5) + c of each 32-column tile.
template <int TM, int TN, bool SWIGLU>
struct AccView32 {
    f32x16_t (&acc)[TN][TM];
    static constexpr int kBlocks = TM;
    static constexpr int kColTiles = SWIGLU ? TN / 2 : TN;
    static constexpr int kCols = kColTiles * 32;
    static constexpr int kGroups = kColTiles * 4;
    __device__ __forceinline__ static int row(int g, int lane) { return lane & 31; }
    __device__ __forceinline__ static int col(int g, int lane) { return (g >> 2) * 32 + 8 * (g & 3) + 4 * (lane >> 5); }
    __device__ __forceinline__ float val(int ib, int g, int c, int half) const {
        return acc[(g >> 2) + half * (TN / 2)][ib][(g & 3) * 4 + c];
    }
};
// 16 x 16 x 32 MFMA: lane holds row (lane & 15), columns 4 (lane >> 4) + c of each 16-column tile; a 32-row
// block is two row tiles.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
template <int TM16, int TN16, bool SWIGLU>
struct AccView16 {
    f32x4_t (&acc)[TN16][TM16];
    static constexpr int kBlocks = TM16 / 2;
    static constexpr int kColTiles = SWIGLU ? TN16 / 2 : TN16;
    static constexpr int kCols = kColTiles * 16;
    static constexpr int kGroups = kColTiles * 2;
    __device__ __forceinline__ static int row(int g, int lane) { return (g / kColTiles) * 16 + (lane & 15); }
    __device__ __forceinline__ static int col(int g, int lane) { return (g % kColTiles) * 16 + 4 * (lane >> 4); }
    __device__ __forceinline__ float val(int ib, int g, int c, int half) const {
        return acc[(g % kColTiles) + half * (TN16 / 2)][2 * ib + g / kColTiles][c];
    }
};

// Epilogue through LDS.  In the accumulator layouts a lane owns 4 consecutive columns of one row,
// so storing straight from registers would issue 8-byte pieces of 64 different cache lines per
// instruction.  Instead every wave transposes 32-row blocks of its sub-tile through a private LDS
// region and writes whole rows: 16 bytes per lane, 128-byte lines fully covered.
// wstage: this wave's private region, 32 * (columns * sizeof(TO) + 16) bytes.
// STREAM: the results leave with non-temporal stores.
// SAVEGU (with SWIGLU): the gate and up accumulators themselves also go to gu[row, col] and gu[row, up_off + col]
// (what the backward pass of a training step needs), through the same staging region.
// DSILU (without SWIGLU): the tile is dh, the gradient of h = silu(g) * u; instead of storing it, every lane reads
// the 16 bytes of g and of u that belong to its 16 bytes of dh (rounded to TO first, as a stored dh would be) from
// gu and stores dg = dh * u * (s + g*s*(1-s)) and du = dh * g * s, s = sigmoid(g), to out[row, col] and
// out[row, up_off + col]: the arithmetic of the elementwise gradient kernel, so the bits are the same.
// tout (SAVEGU or DSILU, 16-bit TO, optional): the same values once more, transposed, for the weight-gradient
// product: tout[col, tcol + row] for the wave's rows, zeros from the group's last row to the next multiple of 64
// (tcol: the wave's first row inside the group + the group's first column; ldt: row stride).  The values are
// staged in a second wave-private LDS region, tstage, with rows along the fast axis:
//   SAVEGU: the accumulator layout already has 16 lanes on 16 consecutive rows, so h goes from the registers
//     into [32 columns][128 rows] (pitch 272 bytes: the lanes of a write land on 64 different banks) and
//     leaves as 256-byte row segments after the last 32-row block;
//   DSILU: dg and du exist only in the row-major phase (a lane holds 8 columns of one row), so two 32-row
//     blocks at a time go into [2][64 columns][64 rows] and leave as whole 128-byte lines (64-byte pieces of
//     lines cost three times as much at the memory side).  That region takes 16 KiB per wave, which fits
//     beside the row-major staging only without padding, so both are unpadded 128-byte rows with XOR swizzles:
//     in the transposed region the 16-byte chunk of a row is XORed with bits 3-5 of the column and columns with
//     bit 2 set trade places with their neighbour (the lanes of a write land on 64 different banks); in the
//     row-major region the chunk is XORed with the low bits of the row.
// In both, two lanes that hold neighbouring rows first exchange half of their values (one DPP move per word), so
// that every LDS write is a whole word holding rows m and m + 1 of one column.
constexpr int kTransPitchH = 128 * 2 + 16;
constexpr int kTransStageH = 32 * kTransPitchH;         // bytes per wave, SAVEGU
constexpr int kTransStageD = 2 * 64 * 128;              // bytes per wave, DSILU
// Bytes of the row-major staging region of one wave.
template <typename TO, typename View, bool DSILU>
constexpr int epilogue_wstage_bytes() {
    return DSILU && sizeof(TO) == 2 && View::kCols == 64 && View::kBlocks == 4
               ? 32 * 128 : 32 * (View::kCols * (int)sizeof(TO) + 16);
}
template <typename TO, typename View, bool SWIGLU, bool SAVEGU = false, bool DSILU = false, bool STREAM = false>
__device__ __forceinline__ void epilogue_view(const View av, unsigned char* wstage, TO* out, int64_t ldo,
                                              int64_t row_base, int rows_valid, int ncol0, int n_out, int lane,
                                              TO* gu = nullptr, int64_t ldgu = 0, int up_off = 0,
                                              TO* tout = nullptr, int64_t ldt = 0, int64_t tcol = 0,
                                              unsigned char* tstage = nullptr) {
    static_assert(!SAVEGU || SWIGLU, "the second output exists for the SwiGLU epilogue only");
    static_assert(!DSILU || !SWIGLU, "the SwiGLU gradient epilogue belongs to the plain product");
    constexpr int WCOLS = View::kCols;
    constexpr int ES = (int)sizeof(TO);
    constexpr bool kSwzStage = DSILU && ES == 2 && WCOLS == 64 && View::kBlocks == 4;   // unpadded, swizzled rows
    constexpr int PITCH = kSwzStage ? 128 : WCOLS * ES + 16;
    static_assert(32 * PITCH == epilogue_wstage_bytes<TO, View, DSILU>(), "staging size");
    constexpr int LPR = WCOLS * ES / 16;   // lanes per output row
    constexpr int RPI = 64 / LPR;          // rows per store instruction
    constexpr int EPC = 16 / ES;           // elements per 16-byte chunk
    constexpr bool kTrans = (SAVEGU || DSILU) && ES == 2 && View::kBlocks * 32 == 128 && (SAVEGU || kSwzStage);
    // rows of the wave that the transposed copy covers: the valid ones and the zero columns after them
    const int t_rows = !kTrans || tout == nullptr || rows_valid <= 0 ? 0
                       : (rows_valid >= 128 ? 128 : (rows_valid + 63) / 64 * 64);
#pragma unroll
    for (int i = 0; i < View::kBlocks; ++i) {
#pragma unroll
        for (int g = 0; g < View::kGroups; ++g) {
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (SWIGLU) v[c] = silu_f(av.val(i, g, c, 0)) * av.val(i, g, c, 1);
                else v[c] = av.val(i, g, c, 0);
            }
            unsigned char* dst = wstage + View::row(g, lane) * PITCH + View::col(g, lane) * ES;
            if constexpr (kSwzStage)
                dst = wstage + View::row(g, lane) * 128 + (((View::col(g, lane) >> 3) ^ (View::row(g, lane) & 7)) * 16) +
                      (View::col(g, lane) & 7) * 2;
            if constexpr (ES == 2) {
                uint2 u;
                u.x = pack_bf16x2(v[0], v[1]);
                u.y = pack_bf16x2(v[2], v[3]);
                *reinterpret_cast<uint2*>(dst) = u;
                if constexpr (kTrans && SAVEGU) {
                    if (t_rows > 0) {
                        // Neighbouring lanes hold neighbouring rows: the even lane takes its neighbour's first two
                        // columns, the odd lane its neighbour's last two, and each writes two whole words (rows m,
                        // m + 1 of one column).
                        const bool odd = (lane & 1) != 0;
                        const uint32_t rcv = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? u.x : u.y), 0xB1, 0xf, 0xf, false);
                        const int m_even = i * 32 + (View::row(g, lane) & ~1);
                        const uint32_t lo = m_even < rows_valid ? (odd ? rcv : u.x) : 0u;
                        const uint32_t hi = m_even + 1 < rows_valid ? (odd ? u.y : rcv) : 0u;
                        unsigned char* td = tstage + (View::col(g, lane) + (odd ? 2 : 0)) * kTransPitchH + m_even * 2;
                        *reinterpret_cast<uint32_t*>(td) = (lo & 0xffffu) | (hi << 16);
                        *reinterpret_cast<uint32_t*>(td + kTransPitchH) = (lo >> 16) | (hi & 0xffff0000u);
                    }
                }
            } else {
                *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int r0 = 0; r0 < 32; r0 += RPI) {
            const int r = r0 + lane / LPR;
            const int c = lane % LPR;
            const u32x4_t data =
                *reinterpret_cast<const u32x4_t*>(wstage + r * PITCH + (kSwzStage ? (c ^ (r & 7)) : c) * 16);
            const int m_local = i * 32 + r;
            const int col = ncol0 + c * EPC;
            if constexpr (DSILU) {
                uint4 pg = make_uint4(0u, 0u, 0u, 0u), pu = make_uint4(0u, 0u, 0u, 0u);
                if (m_local < rows_valid && col < n_out) {
                    const TO* gp = gu + (row_base + m_local) * ldgu + col;
                    TO* dp = out + (row_base + m_local) * ldo + col;
                    float gv[EPC], uv[EPC], dv[EPC], og[EPC], ou[EPC];
                    Elem<TO>::unpack(*reinterpret_cast<const uint4*>(gp), gv);
                    Elem<TO>::unpack(*reinterpret_cast<const uint4*>(gp + up_off), uv);
                    Elem<TO>::unpack(make_uint4(data[0], data[1], data[2], data[3]), dv);
#pragma unroll
                    for (int e = 0; e < EPC; ++e) {
                        const float sg = sigmoid_f(gv[e]);
                        og[e] = dv[e] * uv[e] * (sg + gv[e] * sg * (1.0f - sg));
                        ou[e] = dv[e] * (gv[e] * sg);
                    }
                    pg = Elem<TO>::pack(og);
                    pu = Elem<TO>::pack(ou);
                    *reinterpret_cast<uint4*>(dp) = pg;
                    *reinterpret_cast<uint4*>(dp + up_off) = pu;
                }
                if constexpr (kTrans) {
                    if (i * 32 < t_rows) {
                        // rows past the group's end were left at zero above: they are the zero columns.
                        // Lanes 8 apart hold neighbouring rows of the same 8 columns: the lane of the even row takes
                        // its neighbour's first four columns, the other its neighbour's last four, and each writes
                        // whole words (rows m, m + 1 of one column).
                        const bool odd = (r & 1) != 0;
                        constexpr int kRor8 = 0x128;     // DPP row_ror:8, lane ^ 8 inside a row of 16 lanes
                        const uint32_t rg0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? pg.x : pg.z), kRor8, 0xf, 0xf, false);
                        const uint32_t rg1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? pg.y : pg.w), kRor8, 0xf, 0xf, false);
                        const uint32_t ru0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? pu.x : pu.z), kRor8, 0xf, 0xf, false);
                        const uint32_t ru1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? pu.y : pu.w), kRor8, 0xf, 0xf, false);
                        const uint32_t lo[2][2] = {{odd ? rg0 : pg.x, odd ? rg1 : pg.y}, {odd ? ru0 : pu.x, odd ? ru1 : pu.y}};
                        const uint32_t hi[2][2] = {{odd ? pg.z : rg0, odd ? pg.w : rg1}, {odd ? pu.z : ru0, odd ? pu.w : ru1}};
                        // staged row of column n: n ^ 1 for the columns with bit 2 set (the odd lane's), chunk
                        // (rows / 8 inside the pair of blocks) ^ (n >> 3)
                        const int nb = c * 8 + (odd ? 4 : 0);
                        const int q = (i & 1) * 4 + (r >> 3);
                        unsigned char* td = tstage + ((q ^ c) * 16) + ((r & 7) >> 1) * 4;
#pragma unroll
                        for (int half = 0; half < 2; ++half)
#pragma unroll
                            for (int w2 = 0; w2 < 2; ++w2) {
                                const int n0 = half * 64 + nb + 2 * w2;
                                *reinterpret_cast<uint32_t*>(td + (odd ? n0 + 1 : n0) * 128) =
                                    (lo[half][w2] & 0xffffu) | (hi[half][w2] << 16);
                                *reinterpret_cast<uint32_t*>(td + (odd ? n0 : n0 + 1) * 128) =
                                    (lo[half][w2] >> 16) | (hi[half][w2] & 0xffff0000u);
                            }
                    }
                }
            } else {
                if (m_local < rows_valid && col < n_out) {
                    u32x4_t* const to = reinterpret_cast<u32x4_t*>(out + (row_base + m_local) * ldo + col);
                    if constexpr (STREAM) __builtin_nontemporal_store(data, to);
                    else *to = data;
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if constexpr (kTrans && DSILU) {
            if ((i & 1) && i * 32 < t_rows) {          // t_rows is 64 or 128: both blocks of a pair are in or out
#pragma unroll
                for (int it = 0; it < 16; ++it) {
                    const int idx = it * 64 + lane;
                    const int rowid = idx >> 3, j = idx & 7;          // 128 columns (dg 0..63, du 64..127) x 8 chunks
                    const int n_l = rowid & 63, half = rowid >> 6;
                    const u32x4_t data = *reinterpret_cast<const u32x4_t*>(
                        tstage + (rowid ^ ((rowid >> 2) & 1)) * 128 + ((j ^ ((n_l >> 3) & 7)) * 16));
                    const int m0 = (i - 1) * 32 + j * 8;
                    if (ncol0 + n_l < n_out)
                        __builtin_nontemporal_store(data, reinterpret_cast<u32x4_t*>(tout + (int64_t)(half * up_off + ncol0 + n_l) * ldt + tcol + m0));
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        }
        if constexpr (SAVEGU) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
#pragma unroll
                for (int g = 0; g < View::kGroups; ++g) {
                    unsigned char* dst = wstage + View::row(g, lane) * PITCH + View::col(g, lane) * ES;
                    if constexpr (ES == 2) {
                        uint2 u;
                        u.x = pack_bf16x2(av.val(i, g, 0, half), av.val(i, g, 1, half));
                        u.y = pack_bf16x2(av.val(i, g, 2, half), av.val(i, g, 3, half));
                        *reinterpret_cast<uint2*>(dst) = u;
                    } else {
                        *reinterpret_cast<float4*>(dst) = make_float4(av.val(i, g, 0, half), av.val(i, g, 1, half),
                                                                      av.val(i, g, 2, half), av.val(i, g, 3, half));
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int r0 = 0; r0 < 32; r0 += RPI) {
                    const int r = r0 + lane / LPR;
                    const int c = lane % LPR;
                    const u32x4_t data = *reinterpret_cast<const u32x4_t*>(wstage + r * PITCH + c * 16);
                    const int m_local = i * 32 + r;
                    const int col = ncol0 + c * EPC;
                    if (m_local < rows_valid && col < n_out)
                        *reinterpret_cast<u32x4_t*>(gu + (row_base + m_local) * ldgu + half * up_off + col) = data;
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        }
    }
    if constexpr (kTrans && SAVEGU) {
        if (t_rows > 0) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int r0 = 0; r0 < 32; r0 += 4) {
                const int n_l = r0 + (lane >> 4), ch = lane & 15;
                const u32x4_t data = *reinterpret_cast<const u32x4_t*>(tstage + n_l * kTransPitchH + ch * 16);
                if (ch * 8 < t_rows && ncol0 + n_l < n_out)
                    __builtin_nontemporal_store(data, reinterpret_cast<u32x4_t*>(tout + (int64_t)(ncol0 + n_l) * ldt + tcol + ch * 8));
            }
        }
    }
}

template <typename TO, int TM, int TN, bool SWIGLU, bool SAVEGU = false, bool DSILU = false>
__device__ __forceinline__ void epilogue_staged(f32x16_t (&acc)[TN][TM], unsigned char* wstage, TO* out, int64_t ldo,
                                                int64_t row_base, int rows_valid, int ncol0, int n_out, int lane,
                                                TO* gu = nullptr, int64_t ldgu = 0, int up_off = 0) {
    epilogue_view<TO, AccView32<TM, TN, SWIGLU>, SWIGLU, SAVEGU, DSILU>(AccView32<TM, TN, SWIGLU>{acc}, wstage, out, ldo,
                                                                        row_base, rows_valid, ncol0, n_out, lane, gu,
                                                                        ldgu, up_off);
}

template <typename T, typename TO, int BM, int BN, int WM, int WN, int SM, int SN, bool SWIGLU>
__global__ __launch_bounds__(WM* WN * 64) void grouped_gemm_kernel(GroupedArgs p) {
    constexpr int NT = WM * WN * 64;
    constexpr int VEC = 16 / (int)sizeof(T);
    constexpr int BK = 128 / (int)sizeof(T);
    constexpr int TM = BM / WM / 32;
    constexpr int TN = BN / WN / 32;
    constexpr int RPP = NT / 8;  // rows loaded per pass (8 threads x 16 B per row)
    constexpr int PA = BM / RPP;
    constexpr int PB = BN / RPP;
    constexpr int STAGE = (BM + BN) * kRowPitch;
    static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "wave tiling");
    static_assert(BM % RPP == 0 && BN % RPP == 0, "loader tiling");
    static_assert(!SWIGLU || TN % 2 == 0, "SwiGLU needs gate and up tiles in the same wave");

    extern __shared__ __align__(16) unsigned char smem[];

    TileCoord tc;
    if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc)) return;
    const int count = p.row_count[tc.e];
    const int row0 = p.row_start[tc.e];
    const int K = p.K;
    const T* Bexp = static_cast<const T*>(p.b[tc.e]);
    const T* A = static_cast<const T*>(p.a);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int lrow = tid >> 3;   // loader: row inside a pass
    const int lchunk = tid & 7;  // loader: 16-byte chunk inside the 128-byte slab

    // ---- loader row pointers (nullptr = row does not exist -> zeros)
    const T* ap[PA];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int m = tc.mt * BM + lrow + i * RPP;
        ap[i] = nullptr;
        if (m < count) {
            int64_t src = row0 + m;
            if (p.a_rows) src = p.a_rows[src] / p.a_row_div;
            ap[i] = A + src * p.lda + lchunk * VEC;
        }
    }
    constexpr int HALF = BN / 2;
    const T* bp[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int rb = lrow + i * RPP;
        int n, brow;
        if (SWIGLU) {
            const bool up = rb >= HALF;
            n = tc.nt * HALF + (up ? rb - HALF : rb);
            brow = up ? p.up_offset + n : n;
        } else {
            n = tc.nt * BN + rb;
            brow = n;
        }
        bp[i] = n < p.N_out ? Bexp + (int64_t)brow * p.ldb + lchunk * VEC : nullptr;
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
    u32x4_t ra[PA], rb[PB];

#define ATS_LOAD_GLOBAL(kt_)                                                                       \
    {                                                                                              \
        const int koff = (kt_) * BK;                                                               \
        const bool kok = koff + lchunk * VEC < K;                                                  \
        _Pragma("unroll") for (int i = 0; i < PA; ++i) {                                           \
            ra[i] = zero4;                                                                         \
            if (ap[i] && kok) ra[i] = *reinterpret_cast<const u32x4_t*>(ap[i] + koff);               \
        }                                                                                          \
        _Pragma("unroll") for (int i = 0; i < PB; ++i) {                                           \
            rb[i] = zero4;                                                                         \
            if (bp[i] && kok) rb[i] = *reinterpret_cast<const u32x4_t*>(bp[i] + koff);               \
        }                                                                                          \
    }
#define ATS_STORE_LDS(stage_)                                                                      \
    {                                                                                              \
        unsigned char* sA_ = smem + (stage_) * STAGE;                                              \
        unsigned char* sB_ = sA_ + BM * kRowPitch;                                                 \
        _Pragma("unroll") for (int i = 0; i < PA; ++i)                                             \
            *reinterpret_cast<u32x4_t*>(sA_ + (lrow + i * RPP) * kRowPitch + lchunk * 16) = ra[i];   \
        _Pragma("unroll") for (int i = 0; i < PB; ++i)                                             \
            *reinterpret_cast<u32x4_t*>(sB_ + (lrow + i * RPP) * kRowPitch + lchunk * 16) = rb[i];   \
    }

    // fragment rows of this wave inside the staged tiles
    const int frow = lane & 31;
    const int fgrp = lane >> 5;
    int a_row_off[TM], b_row_off[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_row_off[i] = (wm * (BM / WM) + i * 32 + frow) * kRowPitch + fgrp * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        int r;
        if (SWIGLU) {
            constexpr int WH = BN / WN / 2;  // gate (or up) rows per wave
            r = j < TN / 2 ? wn * WH + j * 32 : HALF + wn * WH + (j - TN / 2) * 32;
        } else {
            r = wn * (BN / WN) + j * 32;
        }
        b_row_off[j] = (r + frow) * kRowPitch + fgrp * 16;
    }

    ATS_LOAD_GLOBAL(0);
    ATS_STORE_LDS(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        if (kt + 1 < nk) ATS_LOAD_GLOBAL(kt + 1);
        const unsigned char* sA = smem + cur * STAGE;
        const unsigned char* sB = sA + BM * kRowPitch;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4_t fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i] = *reinterpret_cast<const u32x4_t*>(sA + a_row_off[i] + ks * 32);
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[j] = *reinterpret_cast<const u32x4_t*>(sB + b_row_off[j] + ks * 32);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) mma_step<T>(fb[j], fa[i], acc[j][i]);
        }
        if (kt + 1 < nk) ATS_STORE_LDS(cur ^ 1);
        __syncthreads();
    }

    // ---- epilogue (all LDS reads of the K loop are behind the last barrier, so LDS is free)
    {
        constexpr int TNO_ = SWIGLU ? TN / 2 : TN;
        constexpr int WSTAGE = 32 * (TNO_ * 32 * (int)sizeof(TO) + 16);
        const int wrow = tc.mt * BM + wm * (BM / WM);
        const int ncol0 = SWIGLU ? tc.nt * HALF + wn * (BN / WN / 2) : tc.nt * BN + wn * (BN / WN);
        epilogue_staged<TO, TM, TN, SWIGLU>(acc, smem + wave * WSTAGE, static_cast<TO*>(p.out), p.ldo,
                                            (int64_t)row0 + wrow, count - wrow, ncol0, p.N_out, lane);
    }
}


// LDS-only barrier: waits for this wave's LDS traffic, not for global loads in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Software-pipelined variant for K % BK == 0.  All loader addresses are valid by
// construction (rows past the end of the expert / of N are clamped; their results are never
// stored), so the steady-state loop body is straight-line code:
//   k-step 0: MFMAs(frag buf 0) while fragments of k-step 1 are read
//   k-step 1: MFMAs(buf 1) | read k-step 2 | slab t+1: registers -> LDS (other stage)
//   k-step 2: MFMAs(buf 0) | read k-step 3 | issue global loads of slab t+2
//   LDS barrier
//   k-step 3: MFMAs(buf 1) | read k-step 0 of slab t+1
// Global loads therefore have a whole slab of MFMA time to land before they are needed.
template <typename T, typename TO, int BM, int BN, int WM, int WN, int SM, int SN, bool SWIGLU, bool WARM,
          bool SLICED = false>
__global__ __launch_bounds__(WM* WN * 64) void grouped_gemm_pipelined_kernel(GroupedArgs p) {
    constexpr int NT = WM * WN * 64;
    constexpr int VEC = 16 / (int)sizeof(T);
    constexpr int BK = 128 / (int)sizeof(T);
    constexpr int TM = BM / WM / 32;
    constexpr int TN = BN / WN / 32;
    constexpr int RPP = NT / 8;
    constexpr int PA = BM / RPP;
    constexpr int PB = BN / RPP;
    constexpr int PITCH = kRowPitch;
    constexpr int STAGE = (BM + BN) * PITCH;
    constexpr int HALF = BN / 2;
    static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "wave tiling");
    static_assert(BM % RPP == 0 && BN % RPP == 0, "loader tiling");
    static_assert(!SWIGLU || TN % 2 == 0, "SwiGLU needs gate and up tiles in the same wave");

    extern __shared__ __align__(16) unsigned char smem[];

    TileCoord tc;
    // SLICED: every expert is k_splits groups, each with a K / k_splits wide slice and its own partial output
    // (without the SwiGLU epilogue only: it is not linear)
    static_assert(!(SLICED && SWIGLU), "slices of K need a linear epilogue");
    constexpr bool sliced = SLICED;
    int split = 0;
    if constexpr (SLICED) {
        if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc, p.k_splits, &split)) return;
        split = __builtin_amdgcn_readfirstlane(split);
    } else {
        if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc)) return;
    }
    const int count = p.row_count[tc.e];
    const int row0 = p.row_start[tc.e];
    const int K = sliced ? p.k_slice : (p.k_count ? p.k_count[tc.e] : p.K);
    const int64_t k_first = sliced ? (int64_t)split * p.k_slice : 0;
    const T* Bexp = static_cast<const T*>(p.b[tc.e]) + k_first;
    const T* A = static_cast<const T*>(p.a_ptrs ? p.a_ptrs[tc.e] : p.a) + k_first;
    const int arow0 = p.a_ptrs ? 0 : row0;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int lrow = tid >> 3;
    const int lchunk = tid & 7;

    const T* ap[PA];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        int m = tc.mt * BM + lrow + i * RPP;
        m = m < count ? m : count - 1;
        int64_t src = arow0 + m;
        if (p.a_rows) src = p.a_rows[src] / p.a_row_div;
        ap[i] = A + src * p.lda + lchunk * VEC;
    }
    const T* bp[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int rb = lrow + i * RPP;
        int n, brow;
        if (SWIGLU) {
            const bool up = rb >= HALF;
            n = tc.nt * HALF + (up ? rb - HALF : rb);
            n = n < p.N_out ? n : p.N_out - 1;
            brow = up ? p.up_offset + n : n;
        } else {
            n = tc.nt * BN + rb;
            n = n < p.N_out ? n : p.N_out - 1;
            brow = n;
        }
        bp[i] = Bexp + (int64_t)brow * p.ldb + lchunk * VEC;
    }

    // L2 warm-up: each thread touches one 128-byte line of a slab that the loaders will ask
    // for kPfDist slabs later, so that the loaders' requests hit in L2.  The values are only
    // folded into a dummy word (which keeps the loads ordered and alive).
    constexpr int kPfDist = 3;
    const T* apf;
    const T* bpf;
    {
        int m = tc.mt * BM + tid % BM;
        m = m < count ? m : count - 1;
        int64_t src = arow0 + m;
        if (p.a_rows) src = p.a_rows[src] / p.a_row_div;
        apf = A + src * p.lda;
        const int rbp = tid % BN;
        int n, brow;
        if (SWIGLU) {
            const bool up = rbp >= HALF;
            n = tc.nt * HALF + (up ? rbp - HALF : rbp);
            n = n < p.N_out ? n : p.N_out - 1;
            brow = up ? p.up_offset + n : n;
        } else {
            n = tc.nt * BN + rbp;
            n = n < p.N_out ? n : p.N_out - 1;
            brow = n;
        }
        bpf = Bexp + (int64_t)brow * p.ldb;
    }
    unsigned pfa[2] = {0u, 0u}, pfb[2] = {0u, 0u}, junk = 0u;

    f32x16_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;

    const int nk = K / BK;
    u32x4_t ra[PA], rb[PB];
    const int st_off = lrow * PITCH + lchunk * 16;

    const int frow = lane & 31;
    const int fgrp = lane >> 5;
    int a_row_off[TM], b_row_off[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
        a_row_off[i] = (wm * (BM / WM) + i * 32 + frow) * PITCH + fgrp * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        int r;
        if (SWIGLU) {
            constexpr int WH = BN / WN / 2;
            r = j < TN / 2 ? wn * WH + j * 32 : HALF + wn * WH + (j - TN / 2) * 32;
        } else {
            r = wn * (BN / WN) + j * 32;
        }
        b_row_off[j] = BM * PITCH + (r + frow) * PITCH + fgrp * 16;
    }
    u32x4_t fa[2][TM], fb[2][TN];

#define PL_LOADG(kt_)                                                                                  \
    {                                                                                                  \
        const int koff = (kt_) * BK;                                                                   \
        _Pragma("unroll") for (int i = 0; i < PA; ++i) ra[i] = *reinterpret_cast<const u32x4_t*>(ap[i] + koff); \
        _Pragma("unroll") for (int i = 0; i < PB; ++i) rb[i] = *reinterpret_cast<const u32x4_t*>(bp[i] + koff); \
    }
#define PL_STORE(stage_)                                                                               \
    {                                                                                                  \
        unsigned char* sA_ = smem + (stage_) * STAGE + st_off;                                         \
        unsigned char* sB_ = sA_ + BM * PITCH;                                                         \
        _Pragma("unroll") for (int i = 0; i < PA; ++i)                                                 \
            *reinterpret_cast<u32x4_t*>(sA_ + i * RPP * PITCH) = ra[i];                                  \
        _Pragma("unroll") for (int i = 0; i < PB; ++i)                                                 \
            *reinterpret_cast<u32x4_t*>(sB_ + i * RPP * PITCH) = rb[i];                                  \
    }
#define PL_READ(stage_, ks_, buf_)                                                                     \
    {                                                                                                  \
        const unsigned char* s_ = smem + (stage_) * STAGE + (ks_) * 32;                                \
        _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                 \
            fa[buf_][i] = *reinterpret_cast<const u32x4_t*>(s_ + a_row_off[i]);                          \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                 \
            fb[buf_][j] = *reinterpret_cast<const u32x4_t*>(s_ + b_row_off[j]);                          \
    }
#define PL_MMA(buf_)                                                                                   \
    {                                                                                                  \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                 \
            _Pragma("unroll") for (int i = 0; i < TM; ++i) mma_step<T>(fb[buf_][j], fa[buf_][i], acc[j][i]); \
    }
// Instruction-order control: inside a phase the scheduler is asked to alternate matrix
// instructions with the memory instructions of that phase (so the memory pipes work in the
// shadow of the MFMAs); nothing moves across a phase boundary.
#define SG_MFMA 0x008
#define SG_VMEM 0x010
#define SG_VMEM_RD 0x020
#define SG_DS_RD 0x100
#define SG_DS_WR 0x200
#define PL_FENCE() __builtin_amdgcn_sched_barrier(0)
#define PL_MIX_READS()                                                                  \
    _Pragma("unroll") for (int g_ = 0; g_ < (TM + TN); ++g_) {                          \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, (TM * TN) / (TM + TN), 0);        \
        __builtin_amdgcn_sched_group_barrier(SG_DS_RD, 1, 0);                           \
    }
#define PL_ITER(kt_, HAS1, HAS2, SLOT)                                                    \
    {                                                                                   \
        const int cur_ = (kt_) & 1;                                                     \
        PL_READ(cur_, 1, 1);                                                            \
        PL_MMA(0);                                                                      \
        PL_MIX_READS();                                                                 \
        PL_FENCE();                                                                     \
        PL_READ(cur_, 2, 0);                                                            \
        if (HAS1) PL_STORE(cur_ ^ 1);                                                   \
        PL_MMA(1);                                                                      \
        if (HAS1) {                                                                     \
            _Pragma("unroll") for (int g_ = 0; g_ < (TM + TN); ++g_) {                  \
                __builtin_amdgcn_sched_group_barrier(SG_MFMA, (TM * TN) / (TM + TN), 0); \
                __builtin_amdgcn_sched_group_barrier(SG_DS_RD, 1, 0);                   \
                __builtin_amdgcn_sched_group_barrier(SG_DS_WR, (PA + PB) / (TM + TN), 0); \
            }                                                                           \
        } else {                                                                        \
            PL_MIX_READS();                                                             \
        }                                                                               \
        PL_FENCE();                                                                     \
        PL_READ(cur_, 3, 1);                                                            \
        if (HAS2) {                                                                     \
            PL_LOADG((kt_) + 2);                                                        \
            if (WARM) {                                                                 \
                junk ^= pfa[SLOT] ^ pfb[SLOT];                                          \
                const int kpf_ = min((kt_) + 2 + kPfDist, nk - 1) * BK;                 \
                pfa[SLOT] = *reinterpret_cast<const unsigned*>(apf + kpf_);             \
                pfb[SLOT] = *reinterpret_cast<const unsigned*>(bpf + kpf_);             \
            }                                                                           \
        }                                                                               \
        PL_MMA(0);                                                                      \
        if (HAS2) {                                                                     \
            _Pragma("unroll") for (int g_ = 0; g_ < (TM + TN); ++g_) {                  \
                __builtin_amdgcn_sched_group_barrier(SG_MFMA, (TM * TN) / (TM + TN), 0); \
                __builtin_amdgcn_sched_group_barrier(SG_DS_RD, 1, 0);                   \
                __builtin_amdgcn_sched_group_barrier(SG_VMEM_RD, (PA + PB) / (TM + TN), 0); \
            }                                                                           \
            if (WARM) __builtin_amdgcn_sched_group_barrier(SG_VMEM_RD, 2, 0);           \
        } else {                                                                        \
            PL_MIX_READS();                                                             \
        }                                                                               \
        PL_FENCE();                                                                     \
        lds_barrier();                                                                  \
        PL_FENCE();                                                                     \
        if (HAS1) PL_READ(cur_ ^ 1, 0, 0);                                              \
        PL_MMA(1);                                                                      \
        if (HAS1) PL_MIX_READS();                                                       \
        PL_FENCE();                                                                     \
    }

    PL_LOADG(0);
    PL_STORE(0);
    if (nk > 1) PL_LOADG(1);
    lds_barrier();
    PL_READ(0, 0, 0);
    int kt = 0;
    for (; kt + 3 < nk; kt += 2) {
        PL_ITER(kt, true, true, 0);
        PL_ITER(kt + 1, true, true, 1);
    }
    if (kt + 2 < nk) {
        PL_ITER(kt, true, true, 0);
        ++kt;
    }
    if (kt + 1 < nk) {
        PL_ITER(kt, true, false, 0);
        ++kt;
    }
    PL_ITER(kt, false, false, 0);
    junk ^= pfa[0] ^ pfb[0] ^ pfa[1] ^ pfb[1];
#undef PL_LOADG
#undef PL_ITER

    TO* out = static_cast<TO*>(p.out) + (sliced ? (int64_t)split * p.part_stride : 0);
    if (p.E < 0) out[0] = TO{};   // never true; with the next line it keeps the warm-up loads alive
    if (p.E < 0 && junk == 0x5a5a5a5au) out[1] = TO{};
    {
        constexpr int TNO_ = SWIGLU ? TN / 2 : TN;
        constexpr int WSTAGE = 32 * (TNO_ * 32 * (int)sizeof(TO) + 16);
        const int wrow = tc.mt * BM + wm * (BM / WM);
        const int ncol0 = SWIGLU ? tc.nt * HALF + wn * (BN / WN / 2) : tc.nt * BN + wn * (BN / WN);
        epilogue_staged<TO, TM, TN, SWIGLU>(acc, smem + wave * WSTAGE, out, p.ldo, (int64_t)row0 + wrow, count - wrow,
                                            ncol0, p.N_out, lane);
    }
}


// Direct-to-LDS variant for K % BK == 0 (bf16 and f32).  The loads write LDS themselves
// (buffer_load_dwordx4 ... lds: lane l of a wave deposits its 16 bytes at M0 + 16*l), so a slab
// never passes through registers: no staging registers, no ds_write instructions.  The loads use
// buffer addressing (descriptor base + 32-bit lane offset + scalar k offset), so advancing along
// K costs no vector ALU work - 64-bit per-lane pointer updates would take issue slots from the
// MFMAs.  The host only selects this kernel when every lane offset fits in 32 bits.
//
// One wave instruction fills 1 KiB = 8 rows x 128 bytes, rows unpadded.  Bank conflicts on the
// fragment reads are avoided by an XOR swizzle applied on the global side: LDS slot s of row R
// holds the 16-byte chunk  s ^ f(R),  f(R) = (R & 7) ^ ((R >> 3) & 1), and a reader that wants
// chunk c of row R reads slot c ^ f(R).  For the 16 consecutive rows that one quarter-wave reads,
// (R & 1, c ^ f(R)) takes 16 different values, i.e. all 64 banks are hit once.
//
// LDS map: [A stage 0][A stage 1][A stage 2][B stage 0][B stage 1] (160 KiB for the 256 x 256 tile).  The
// activation slabs go round a ring of three stages, the weight slabs alternate between two:
// after the barrier that ends slab t, the weight loads of slab t+2 (into the stage slab t used) and the
// activation loads of slab t+3 are issued, in that order.  The weight loads have one slab of MFMA time to
// land, the activation loads two, and the wait at the end of a slab lets the youngest activation loads stay
// in flight (s_waitcnt vmcnt(NIA)): only half of a slab's loads sit in the window that the barrier closes,
// so the burst that the address unit has to work off after every barrier is halved.
// The weight stage is a compile-time offset of the read instructions; the activation stage is a scalar
// that is added to the fragment address once per k-step.
//
// Schedule per slab t (4 k-steps of MFMAs, fragments double buffered in registers):
//   k-steps 0..2 : MFMAs | fragment reads of the next k-step
//   wait for the loads of slab t+1, barrier (every wave is done reading slab t)
//   issue the loads (weights of slab t+2, activations of slab t+3)
//   k-step 3     : MFMAs | fragment reads of k-step 0 of slab t+1
template <typename T, typename TO, int BM, int BN, int WM, int WN, int SM, int SN, bool SWIGLU, bool SAVEGU = false,
          bool DSILU = false>
__global__ __launch_bounds__(WM* WN * 64) void grouped_gemm_dma_kernel(GroupedArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int NW = WM * WN;
    constexpr int ES = (int)sizeof(T);
    constexpr int TM = BM / WM / 32;
    constexpr int TN = BN / WN / 32;
    constexpr int NIA = BM / 8 / NW;  // load instructions per wave and slab, A rows
    constexpr int NIB = BN / 8 / NW;
    constexpr int HALF = BN / 2;
    constexpr int A_STAGE = BM * 128;
    constexpr int B_STAGE = BN * 128;
    constexpr int B_BASE = 3 * A_STAGE;
    static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "wave tiling");
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && NW % 2 == 0, "loader tiling");
    static_assert(!SWIGLU || TN % 2 == 0, "SwiGLU needs gate and up tiles in the same wave");
    static_assert((TM - 1) * 4096 + 128 <= 65536 && B_STAGE + (BN / 2 + 32 * TN) * 128 <= 65536, "offset field");

    extern __shared__ __align__(16) unsigned char smem[];
    typedef __attribute__((address_space(3))) void* lds_ptr_t;

    TileCoord tc;
    if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc)) return;
    const int count = p.row_count[tc.e];
    const int row0 = p.row_start[tc.e];
    const int K = p.k_count ? p.k_count[tc.e] : p.K;
    const T* Bexp = static_cast<const T*>(p.b[tc.e]);
    const T* A = static_cast<const T*>(p.a_ptrs ? p.a_ptrs[tc.e] : p.a);
    const int arow0 = p.a_ptrs ? 0 : row0;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;

    // ---- load descriptors and lane offsets: instruction j of this wave covers rows (j*NW + wave)*8 .. +8
    constexpr int kRsrcFlags = 0x00020000;  // raw buffer, 32-bit data format
    const bool gather = p.a_rows != nullptr;
    // without a gather the A descriptor starts at the tile's first row, so lane offsets stay small
    const T* a_base = gather ? A : A + ((int64_t)arow0 + (int64_t)tc.mt * BM) * p.lda;
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a_base), 0, (int)p.a_extent_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(Bexp), 0, (int)p.b_extent_bytes, kRsrcFlags);
    const int drow = lane >> 3;                         // row inside the 8-row group
    const int dchunk = (lane & 7) ^ drow ^ (wave & 1);  // global chunk that lands in slot lane&7
    unsigned ao[NIA], bo[NIB];
#pragma unroll
    for (int j = 0; j < NIA; ++j) {
        int m = tc.mt * BM + (j * NW + wave) * 8 + drow;
        m = m < count ? m : count - 1;
        int64_t src = gather ? (int64_t)(p.a_rows[arow0 + m] / p.a_row_div) : (int64_t)(m - tc.mt * BM);
        ao[j] = (unsigned)(src * p.lda * ES + dchunk * 16);
    }
#pragma unroll
    for (int j = 0; j < NIB; ++j) {
        const int rb = (j * NW + wave) * 8 + drow;
        int n, brow;
        if (SWIGLU) {
            const bool up = rb >= HALF;
            n = tc.nt * HALF + (up ? rb - HALF : rb);
            n = n < p.N_out ? n : p.N_out - 1;
            brow = up ? p.up_offset + n : n;
        } else {
            n = tc.nt * BN + rb;
            n = n < p.N_out ? n : p.N_out - 1;
            brow = n;
        }
        bo[j] = (unsigned)((int64_t)brow * p.ldb * ES + dchunk * 16);
    }
    unsigned char* const dma_a = smem + wave * 1024;           // + stage*A_STAGE + j*NW*1024
    unsigned char* const dma_b = smem + B_BASE + wave * 1024;  // + stage*B_STAGE + j*NW*1024

    f32x16_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;

    const int nk = K * ES / 128;

    // ---- fragment addresses: one register per k-step and operand; rows and stages by offset
    const int frow = lane & 31;
    const int fgrp = lane >> 5;
    const int fsw = fgrp ^ (frow & 7) ^ ((frow >> 3) & 1);
    const unsigned char* fa_addr[4];
    const unsigned char* fb_addr[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int slot = (2 * ks) ^ fsw;
        fa_addr[ks] = smem + (wm * (BM / WM) + frow) * 128 + slot * 16;
        fb_addr[ks] = smem + B_BASE + (wn * (SWIGLU ? BN / WN / 2 : BN / WN) + frow) * 128 + slot * 16;
    }
    u32x4_t fa[2][TM], fb[2][TN];

#define DM_ISSUE_A(kt_, aoff_)                                                                         \
    {                                                                                                  \
        const int soff = (kt_) * 128;                                                                  \
        _Pragma("unroll") for (int j = 0; j < NIA; ++j)                                                \
            __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                  \
                rsrc_a, (lds_ptr_t)(dma_a + (aoff_) + j * NW * 1024), 16, ao[j], soff, 0, 0);          \
    }
#define DM_ISSUE_B(kt_, stage_)                                                                        \
    {                                                                                                  \
        const int soff = (kt_) * 128;                                                                  \
        _Pragma("unroll") for (int j = 0; j < NIB; ++j)                                                \
            __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                  \
                rsrc_b, (lds_ptr_t)(dma_b + (stage_) * B_STAGE + j * NW * 1024), 16, bo[j], soff, 0, 0); \
    }
#define DM_B_ROW(j_) (SWIGLU ? ((j_) < TN / 2 ? (j_) * 32 : HALF + ((j_) - TN / 2) * 32) : (j_) * 32)
// Read order = use order of the MFMAs (weight fragment 0, all activation fragments, then the
// other weight fragments), so the first MFMAs of the next k-step wait for few reads.
#define DM_READ(aoff_, stage_, ks_, buf_)                                                              \
    {                                                                                                  \
        const unsigned char* fa_ = fa_addr[ks_] + (aoff_);                                             \
        fb[buf_][0] = *reinterpret_cast<const u32x4_t*>(fb_addr[ks_] + (stage_) * B_STAGE + DM_B_ROW(0) * 128); \
        _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                 \
            fa[buf_][i] = *reinterpret_cast<const u32x4_t*>(fa_ + i * 4096);                           \
        _Pragma("unroll") for (int j = 1; j < TN; ++j)                                                 \
            fb[buf_][j] = *reinterpret_cast<const u32x4_t*>(fb_addr[ks_] + (stage_) * B_STAGE + DM_B_ROW(j) * 128); \
    }
// k-step 3: the fragment reads go first (one per MFMA), the loads fill the remaining slots.
#define DM_MIX_DMA()                                                                    \
    _Pragma("unroll") for (int g_ = 0; g_ < (TM + TN); ++g_) {                          \
        __builtin_amdgcn_sched_group_barrier(SG_DS_RD, 1, 0);                           \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);                            \
        __builtin_amdgcn_sched_group_barrier(SG_VMEM, 1, 0);                            \
    }                                                                                   \
    _Pragma("unroll") for (int g_ = 0; g_ < TM * TN - (TM + TN); ++g_) {                \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);                            \
        __builtin_amdgcn_sched_group_barrier(SG_VMEM, 1, 0);                            \
    }
// STG: weight stage of slab kt (compile time); sa_cur / sa_nxt: activation stage offsets of slabs kt and
// kt+1.  Slabs past the end are clamped to the last one: their loads land in stages nobody reads again,
// which keeps the loop body free of special cases.
#define DM_ITER(kt_, STG)                                                               \
    {                                                                                   \
        DM_READ(sa_cur, STG, 1, 1);                                                     \
        PL_MMA(0);                                                                      \
        PL_MIX_READS();                                                                 \
        PL_FENCE();                                                                     \
        DM_READ(sa_cur, STG, 2, 0);                                                     \
        PL_MMA(1);                                                                      \
        PL_MIX_READS();                                                                 \
        PL_FENCE();                                                                     \
        DM_READ(sa_cur, STG, 3, 1);                                                     \
        PL_MMA(0);                                                                      \
        PL_MIX_READS();                                                                 \
        PL_FENCE();                                                                     \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NIA) : "memory"); \
        PL_FENCE();                                                                     \
        DM_READ(sa_nxt, STG ^ 1, 0, 0);                                                 \
        DM_ISSUE_B(min((kt_) + 2, nk - 1), STG);                                        \
        DM_ISSUE_A(min((kt_) + 3, nk - 1), sa_cur);                                     \
        PL_MMA(1);                                                                      \
        DM_MIX_DMA();                                                                   \
        PL_FENCE();                                                                     \
        sa_cur = sa_nxt;                                                                \
        sa_nxt = sa_nxt == 2 * A_STAGE ? 0 : sa_nxt + A_STAGE;                          \
    }

    DM_ISSUE_A(0, 0);
    DM_ISSUE_B(0, 0);
    DM_ISSUE_A(min(1, nk - 1), A_STAGE);
    DM_ISSUE_B(min(1, nk - 1), 1);
    DM_ISSUE_A(min(2, nk - 1), 2 * A_STAGE);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NIA + NIB) : "memory");
    int sa_cur = 0, sa_nxt = A_STAGE;
    DM_READ(sa_cur, 0, 0, 0);
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        DM_ITER(kt, 0);
        DM_ITER(kt + 1, 1);
    }
    if (kt < nk) DM_ITER(kt, 0);
    // the clamped loads of the last slabs may still be in flight; the epilogue reuses LDS
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#undef DM_ISSUE_A
#undef DM_ISSUE_B
#undef DM_READ
#undef DM_ITER
#undef DM_B_ROW
#undef DM_MIX_DMA

    {
        constexpr int TNO_ = SWIGLU ? TN / 2 : TN;
        constexpr int WSTAGE = 32 * (TNO_ * 32 * (int)sizeof(TO) + 16);
        const int wrow = tc.mt * BM + wm * (BM / WM);
        const int ncol0 = SWIGLU ? tc.nt * HALF + wn * (BN / WN / 2) : tc.nt * BN + wn * (BN / WN);
        epilogue_staged<TO, TM, TN, SWIGLU, SAVEGU, DSILU>(acc, smem + wave * WSTAGE, static_cast<TO*>(p.out), p.ldo,
                                                    (int64_t)row0 + wrow, count - wrow, ncol0, p.N_out, lane,
                                                    static_cast<TO*>(p.gu_out), p.ld_gu, p.up_offset);
    }
#endif
}

// bf16 prefill tile on v_mfma_f32_16x16x32_bf16.  Same data movement as grouped_gemm_dma_kernel (256 x 256 tile,
// 8 waves of 128 x 64, direct-to-LDS slabs, three activation stages and two weight stages), but the products
// are formed by the 16 x 16 x 32 instruction: with random bf16 operands the chip, which is power limited on this
// kernel, sustains about 14 % more of them per second than of the 32 x 32 x 16 form (measured on MFMA-only loops:
// 2.13 vs 1.86 PFLOP/s).
// Swizzle: slot s of row R holds chunk s ^ (R & 7).  A fragment read has lane l on row l % 16 and chunk
// 4 ks + l / 16; measured with the bank-conflict counter on a stand-alone kernel that issues only this read, the
// hardware serves it in 4 cycles (no conflict), while the f(R) = (R & 7) ^ ((R >> 3) & 1) of the 32 x 32 x 16 kernel,
// which a model of 16 consecutive lanes per cycle prefers, takes 8 (SQ_LDS_BANK_CONFLICT = half of
// SQ_LDS_IDX_ACTIVE, also over the whole GEMM launch): the lanes that share a cycle are not 16 consecutive ones.
// LDS was busy 60 % of this kernel's cycles with that conflict; without it the prefill step is 0.45 % faster.
//
// MIDROWS: the instance for groups of a few hundred rows.  A group is cut into as few tiles as possible, all of one
// height (a multiple of 16 rows), and a tile's rows are dealt to the two wave rows, which differ by one fragment where their
// number is odd: a SIMD has a wave of each, so every SIMD has the same, smallest number of MFMAs (heights in steps of 32
// instead of 16: 8 experts with 358-407 rows each, gate/up 603 against 584 us, down 292 against 288); with 256-row tiles and the rest, a group of 192 rows kept one wave of a SIMD at 128
// rows beside one at 64.  There the weights also come from HBM instead of from the L2 of an XCD that four or more
// row tiles share, so the three-stage ring is the weights' and the activations have the two stages (the roles in
// the phases below trade places).  Rows per group, gate/up [28672, 4096] x 8 | down [4096, 14336] x 8 | gate/up
// [2816, 2048] x 64, microseconds, before -> now (the second figure: equal heights, but the ring for the activations):
//   192   569 -> 425 -> 426  |  262 -> 259 -> 261  |  236 -> 187 -> 187
//   320   601 -> 588 -> 571  |  307 -> 299 -> 283  |  275 -> 276 -> 272
//   383   642 -> 635 -> 622  |  324 -> 314 -> 306  |  286 -> 295 -> 287
//   1024 1469 -> 1498 -> 1493 |  815 -> 819 -> 819 |  629 -> 641 -> 639
//   4096 5473 -> 5520 -> 5556 | 2734 -> 2765 -> 2773 | 2380 -> 2413 -> 2442
// and on another card (full height, this form)
//   448   674, 673  |  320, 313  |  301, 302          640  1014, 1020  |  575, 562  |  431, 433
//   512   727, 736  |  334, 337  |  322, 327          704  1062, 1101  |  600, 618  |  451, 473
//   576   981, 937  |  548, 523  |  413, 399          768  1121, 1120  |  614, 613  |  480, 479
// It gains where a group's last full-height tile would be half empty or more, loses up to 4 % where that is nearly full, and
// among groups of unequal size evens out between 512 and 768.  So launches below kMidRowsMaxAvg rows per group take it,
// and those of one group at any height that dense_tile_rows finds.
// Sums over K are in the same order in both instances.
//
// A 64-element slab is two 32-element k-steps; the wave's rows are up to two halves of up to four 16-row fragments.
// A slab is four phases of up to 16 MFMAs, (k-step, row half) = (0,0) (0,1) (1,0) (1,1); fragments live in two
// buffers of four activation fragments and two buffers of four weight fragments:
//   phase 0 : MFMAs | reads: activations (k0, half 1), weights (k1) 0..1 | loads: activations of slab t+2, 1 of 4
//   phase 1 : MFMAs | reads: activations (k1, half 0), weights (k1) 2..3 | loads: activations of slab t+2, 1 of 4
//   phase 2 : MFMAs | reads: activations (k1, half 1)                    | loads: activations of slab t+2, 2 of 4
//   wait for the loads of slab t+1, barrier
//   phase 3 : MFMAs | reads: activations (k0, half 0) and weights (k0) of slab t+1 | loads: weights of slab t+2
// The activation ring has three stages, so the stage that slab t+2 goes into was given up at the previous
// barrier and its loads can be issued anywhere in slab t; the weights have two stages, so theirs have to
// follow the barrier.  With all eight loads of a wave behind the barrier the 64 loads of the workgroup
// reached the texture addresser within a few hundred cycles, its queue filled up (it takes one 1 KiB load in
// about 16 cycles) and the waves, which issue in order, stood at their next load with MFMAs behind it:
// spreading the activation loads over the slab is worth 3-4 % at the prefill and at the fine-grained shape.
// Inside a phase the fragment reads go between its first MFMAs and the loads between the MFMAs behind them
// (in phase 3: eight reads over the first eight MFMAs, four loads over the last eight).  With the loads at the
// head of their phase, next to the reads, the prefill step was 3.3 % slower and the training step 3.4 %
// (alternating runs on one box: 5.70 -> 5.51 ms and 19.69 -> 19.03 ms); loads of one array bunched into one
// phase, or weight loads held back until after the next slab has begun, lose it again.
// A wave runs phase 3 (the weight loads of slab t+2 and the first fragment reads of slab t+1, right behind the
// barrier) at raised priority and drops back at the top of the next slab: 1 % at both shapes and on the training
// step (s_setprio 1, 2 or 3, and keeping it through phase 0, measure the same at the prefill shape; raising it for
// phases 0-2 instead loses 0.2 %); with the order of reads and loads described above it is worth 2.5 % (5.81 against
// 5.66 ms without / with it).
//
// BKM: the weight operand is stored [K][N] (K-major: the reduction index walks rows of p.ldb elements) instead
// of [N][K].  That is the layout of the forward's own weights as the backward's data gradients need them
// (dx = dy . W with W [N_fwd = K][K_fwd = N]), so no transposed copy of the weights is made per step.  A slab of
// it is 64 rows of 256 output columns (512 bytes, again 32 KiB a stage); a weight fragment (16 output columns x
// 32 reduction steps) comes out through the transposing read ds_read_b64_tr_b16: a group of 16 lanes reads a
// block of 4 rows x 32 bytes and lane i receives its column i, two reads give a lane its 8 consecutive reduction
// steps - the same register contents as the 16-byte read of the [N][K] layout, so both layouts give the same
// bits.  The 32-byte chunks of a row are swizzled on the global side, chunk c of stage row r lands in slot
// c ^ f(r), f(r) = (r % 4) | ((r / 8) % 4) << 2: the 16 row pieces that one read instruction touches fall on 16
// different slots, i.e. on all banks once.
//
// AKM: the other operand is stored [K][rows] as well (one group; p.b is the operand itself, p.K its exact number of rows): the
// weight gradient of a linear layer from the gradients and activations as they lie, tokens along the rows, without
// transposed copies.  The same slabs, swizzle and transposing reads; same bits as the product of transposed copies.
//
// ONCE: groups of one tile each, whose weights are read from HBM by nobody else: loaded non-temporally, and in the gate/up product eight
// supertiles in turn begin K an eighth of it apart and come round (its rows of 4 and 8 KB put a column of all of them into a few of the
// memory's channels; the down projections' gain nothing).  Where every group has its tile these are the eight XCDs, each in step by
// itself; the start follows from expert and columns alone, so that the order of a row's sums does not depend on the other groups.
// Layers, microseconds, as the instance for every group -> non-temporal -> out of step: 8 experts top-2 of [28672, 4096], 550 tokens
// 610 -> 572 -> 559, 700 642 -> 597 -> 586, 890 690 -> 640 -> 633; 64 experts top-6 of [2816, 2048], 1500 tokens 309 -> 297 -> 291, 2200
// 338 -> 319 -> 313.  Where groups reach a second tile it costs what it gained: 1100 tokens of 8 experts 868 -> 873, 3000 of 64 448 ->
// 459, hence kOnceMaxAvgRows.
template <typename TO, int SM, int SN, bool SWIGLU, bool SAVEGU = false, bool DSILU = false, bool BKM = false,
          bool MIDROWS = false, bool SLICED = false, bool AKM = false, bool ONCE = false>
__device__ __forceinline__ void grouped_gemm_dma16_body(const GroupedArgs& p, unsigned char* smem,
                                                         const int32_t* __restrict__ row_count) {
#if defined(__HIP_DEVICE_COMPILE__)
    static_assert(!BKM || (!SWIGLU && !SAVEGU), "the K-major weight layout serves the plain product and the dgrad epilogue");
    static_assert(!SLICED || (MIDROWS && !SWIGLU && !DSILU), "slices of K need a linear epilogue");
    static_assert(!AKM || (BKM && MIDROWS && !DSILU), "both operands K-major: the plain product in tiles of equal height");
    typedef bf16_t T;
    constexpr int BM = 256, BN = 256, WM = 2, WN = 4;
    constexpr int NW = WM * WN;
    constexpr int ES = 2;
    constexpr int TM = 8;   // 16-row activation fragments per wave
    constexpr int TN = 4;   // 16-row weight fragments per wave
    constexpr int NIA = BM / 8 / NW;
    constexpr int NIB = BN / 8 / NW;
    constexpr int HALF = BN / 2;
    constexpr int A_STAGE = BM * 128;
    constexpr int B_STAGE = BN * 128;
    constexpr int B_BASE = (MIDROWS ? 2 : 3) * A_STAGE;
    static_assert(A_STAGE == B_STAGE, "the two rings share their stage offsets");

    typedef __attribute__((address_space(3))) void* lds_ptr_t;

    TileCoord tc;
    const int most_rows = MIDROWS && p.tile_rows ? p.tile_rows : BM;
    int split = 0;                      // slice of K of this tile
    if constexpr (SLICED) {
        if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, most_rows, p.n_tiles, p.sm, p.sn, false, &tc, p.k_splits, &split)) return;
        split = __builtin_amdgcn_readfirstlane(split);
    } else {
        if (!decode_tile_wave(blockIdx.x, p.row_count, p.E, most_rows, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0, &tc)) return;
    }
    const int count = row_count[tc.e];
    const int row0 = p.row_start[tc.e];
    const int64_t k_first = SLICED ? (int64_t)split * p.k_slice : 0;
    const int K = AKM ? (int)(SLICED && k_first + p.k_slice < p.K ? p.k_slice : p.K - k_first)
                  : SLICED ? p.k_slice : p.k_count ? p.k_count[tc.e] : p.K;
    const T* Bexp = (AKM ? reinterpret_cast<const T*>(p.b) : static_cast<const T*>(p.b[tc.e])) + (BKM ? k_first * p.ldb : k_first);
    const T* A = static_cast<const T*>(p.a_ptrs ? p.a_ptrs[tc.e] : p.a) + (AKM ? k_first * p.lda : k_first);
    const int arow0 = p.a_ptrs ? 0 : row0;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;

    // ---- rows of this tile: the upper wave row takes the first share of them, the lower one the rest
    int frags = TM;                     // 16-row fragments of this wave
    int share0 = 128, share1 = 128;     // rows of the two wave rows
    if constexpr (MIDROWS) {
        const int m_tiles = (count + most_rows - 1) / most_rows;
        const int f = __builtin_amdgcn_readfirstlane(((count + m_tiles - 1) / m_tiles + 15) / 16);
        share0 = (f + 1) / 2 * 16;
        share1 = f > 1 ? f / 2 * 16 : 16;
        frags = (wm == 0 ? share0 : share1) / 16;
    }
    const int tile_row = tc.mt * (share0 + share1);

    // ---- load descriptors and lane offsets: instruction j of this wave covers rows (j*NW + wave)*8 .. +8
    constexpr int kRsrcFlags = 0x00020000;  // raw buffer, 32-bit data format
    const bool gather = p.a_rows != nullptr;
    const T* a_base = gather || AKM ? A : A + ((int64_t)arow0 + (int64_t)tile_row) * p.lda;
    // AKM: the descriptors end with the last of the K rows, what lies behind it reads as zero
    const uint32_t a_extent = AKM ? (uint32_t)(((int64_t)(K - 1) * p.lda + count) * ES) : p.a_extent_bytes;
    const uint32_t b_extent = AKM ? (uint32_t)(((int64_t)(K - 1) * p.ldb + p.N_out) * ES) : p.b_extent_bytes;
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a_base), 0, (int)a_extent, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(Bexp), 0, (int)b_extent, kRsrcFlags);
    const int drow = lane >> 3;
    const int dchunk = (lane & 7) ^ drow;
    unsigned ao[NIA], bo[NIB];
    // the gather indices are asked for first: the weight loads issued below are in flight while they arrive
    int a_idx[NIA];
#pragma unroll
    for (int j = 0; j < NIA; ++j) {
        if constexpr (AKM) {
            // as the K-major weights below, columns 0 .. 127 of a stage for wave row 0, the others for wave row 1
            const int r = 2 * (j * NW + wave) + (lane >> 5);
            const int f = (r & 3) | (((r >> 3) & 3) << 2);
            const int col = ((lane & 31) ^ (f << 1)) * 8;
            int m = (col & 127) < (col < 128 ? share0 : share1) ? tile_row + (col >> 7) * share0 + (col & 127) : count - 8;
            m = m <= count - 8 ? m : count - 8;
            ao[j] = (unsigned)(((int64_t)r * p.lda + m) * ES);
            continue;
        }
        // stage rows 0 .. 127 belong to wave row 0, the others to wave row 1; rows that nobody has repeat the last one
        const int r = (j * NW + wave) * 8 + drow;
        int m = (r & 127) < (r < 128 ? share0 : share1) ? tile_row + (r >> 7) * share0 + (r & 127) : count - 1;
        m = m < count ? m : count - 1;
        a_idx[j] = gather ? p.a_rows[arow0 + m] : m - tile_row;
    }
#pragma unroll
    for (int j = 0; j < NIB; ++j) {
        if constexpr (BKM) {
            // instruction j of this wave fills stage rows 2 (j NW + wave), + 1: lane l the 16 bytes l % 32 of row l / 32
            const int r = 2 * (j * NW + wave) + (lane >> 5);
            const int f = (r & 3) | (((r >> 3) & 3) << 2);
            int n = tc.nt * BN + ((lane & 31) ^ (f << 1)) * 8;
            n = n <= p.N_out - 8 ? n : p.N_out - 8;      // columns past the end repeat the last eight (never stored)
            bo[j] = (unsigned)(((int64_t)r * p.ldb + n) * ES);
            continue;
        }
        const int rb = (j * NW + wave) * 8 + drow;
        int n, brow;
        if (SWIGLU) {
            const bool up = rb >= HALF;
            n = tc.nt * HALF + (up ? rb - HALF : rb);
            n = n < p.N_out ? n : p.N_out - 1;
            brow = up ? p.up_offset + n : n;
        } else {
            n = tc.nt * BN + rb;
            n = n < p.N_out ? n : p.N_out - 1;
            brow = n;
        }
        bo[j] = (unsigned)((int64_t)brow * p.ldb * ES + dchunk * 16);
    }
    unsigned char* const dma_a = smem + wave * 1024;
    unsigned char* const dma_b = smem + B_BASE + wave * 1024;

    f32x4_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int nk = AKM ? (K + 63) / 64 : K * ES / 128;

    // ---- fragment addresses: one register per k-step and operand; fragments and weight stages by offset
    const int frow = lane & 15;
    const int kgrp = lane >> 4;
    const int fsw = frow & 7;
    const unsigned char* fa_addr[2];
    const unsigned char* fb_addr[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const int slot = (4 * ks + kgrp) ^ fsw;
        fa_addr[ks] = smem + (wm * (BM / WM) + frow) * 128 + slot * 16;
        fb_addr[ks] = smem + B_BASE + (wn * (SWIGLU ? BN / WN / 2 : BN / WN) + frow) * 128 + slot * 16;
    }
    // K-major weights: fragment j of a k-step sits in slot ((wn ^ q) << 2 | (j ^ t)) of rows 8 q + t (+ 4), lane
    // 16 q + i, t = i / 4, 8 (i % 4) bytes in; k-step and stage are immediate offsets
    typedef short tr4_t __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) tr4_t* lds_tr_ptr_t;
    typedef __attribute__((address_space(3))) unsigned char* lds_u8_t;
    lds_u8_t fb_tr[TN], fa_tr[AKM ? TM : 1];
    if constexpr (AKM) {      // fragment i of a wave's eight: column block 8 wm + i
        const int t4 = frow >> 2;
#pragma unroll
        for (int i = 0; i < TM; ++i)
            fa_tr[i] = (lds_u8_t)smem + (8 * kgrp + t4) * 512 + 8 * (frow & 3) +
                       (((((2 * wm + (i >> 2)) ^ kgrp) & 3) << 2) | ((i & 3) ^ t4)) * 32;
    }
    if constexpr (BKM) {
        const int t4 = frow >> 2;
        const int base0 = B_BASE + (8 * kgrp + t4) * 512 + 8 * (frow & 3) + (((wn ^ kgrp) & 3) << 2) * 32;
#pragma unroll
        for (int j = 0; j < TN; ++j) fb_tr[j] = (lds_u8_t)smem + base0 + ((j ^ t4) * 32);
    }
    // bytes from one slab of an operand to the next (unsigned: the advance along K runs up to 4 GiB)
    const unsigned b_slab = BKM ? (unsigned)(p.ldb * 128) : 128u;
    const unsigned a_slab = AKM ? (unsigned)(p.lda * 128) : 128u;
    constexpr int RB2 = BKM ? 4 : 2;   // read instructions of two weight fragments
    constexpr int RA = AKM ? 2 : 1;    // read instructions of an activation fragment
    u32x4_t fa[2][4], fb[2][TN];

// AKM: the advance along K is part of the lane offset, which the descriptor's end is checked against (the scalar offset is
// not); otherwise it is the scalar offset.
#define D16_LOAD(rsrc_, dst_, off_, adv_, policy_)                                                     \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_, (lds_ptr_t)(dst_), 16, (off_) + (AKM ? (adv_) : 0u), \
                                             AKM ? 0 : (int)(adv_), 0, policy_)
#define D16_ISSUE_A1(kt_, aoff_, j_) D16_LOAD(rsrc_a, dma_a + (aoff_) + (j_) * NW * 1024, ao[j_], (unsigned)(kt_) * a_slab, 0)
#define D16_ISSUE_B1(kt_, boff_, j_) \
    D16_LOAD(rsrc_b, dma_b + (boff_) + (j_) * NW * 1024, bo[j_], (unsigned)(kt_) * b_slab, ONCE ? kNonTemporal : 0)
#define D16_ISSUE_A(kt_, aoff_)                                                                        \
    {                                                                                                  \
        const unsigned adv = (unsigned)(kt_) * a_slab;                                                  \
        _Pragma("unroll") for (int j = 0; j < NIA; ++j)                                                \
            D16_LOAD(rsrc_a, dma_a + (aoff_) + j * NW * 1024, ao[j], adv, 0);                          \
    }
#define D16_ISSUE_B(kt_, boff_)                                                                        \
    {                                                                                                  \
        const unsigned adv = (unsigned)(kt_) * b_slab;                                                  \
        _Pragma("unroll") for (int j = 0; j < NIB; ++j)                                                \
            D16_LOAD(rsrc_b, dma_b + (boff_) + j * NW * 1024, bo[j], adv, ONCE ? kNonTemporal : 0);    \
    }
#define D16_B_ROW(j_) (SWIGLU ? ((j_) < TN / 2 ? (j_) * 16 : HALF + ((j_) - TN / 2) * 16) : (j_) * 16)
#define D16_READ_A(aoff_, ks_, f0_, nf_, buf_)                                                         \
    if constexpr (AKM) {                                                                               \
        _Pragma("unroll") for (int i = 0; i < (nf_); ++i) {                                            \
            union {                                                                                    \
                tr4_t t[2];                                                                            \
                u32x4_t u;                                                                             \
            } cv_;                                                                                     \
            const lds_u8_t pa_ = fa_tr[(AKM ? (f0_) + i : 0)] + (aoff_) + (ks_) * (32 * 512);          \
            cv_.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr_t)(pa_));                   \
            cv_.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr_t)(pa_ + 4 * 512));         \
            fa[buf_][i] = cv_.u;                                                                       \
        }                                                                                              \
    } else {                                                                                                  \
        const unsigned char* fa_ = fa_addr[ks_] + (aoff_) + (f0_) * 2048;                              \
        _Pragma("unroll") for (int i = 0; i < (nf_); ++i)                                              \
            fa[buf_][i] = *reinterpret_cast<const u32x4_t*>(fa_ + i * 2048);                           \
    }
#define D16_READ_B(boff_, ks_, j_, buf_)                                                               \
    if constexpr (BKM) {                                                                               \
        union {                                                                                        \
            tr4_t t[2];                                                                                \
            u32x4_t u;                                                                                 \
        } cv_;                                                                                         \
        const lds_u8_t pb_ = fb_tr[j_] + (boff_) + (ks_) * (32 * 512);                      \
        cv_.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr_t)(pb_));                       \
        cv_.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr_t)(pb_ + 4 * 512));             \
        fb[buf_][j_] = cv_.u;                                                                          \
    } else                                                                                             \
        fb[buf_][j_] = *reinterpret_cast<const u32x4_t*>(fb_addr[ks_] + (boff_) + D16_B_ROW(j_) * 128)
#define D16_MMA(bbuf_, abuf_, f0_, nf_)                                                                 \
    {                                                                                                  \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                 \
            _Pragma("unroll") for (int i = 0; i < (nf_); ++i) {                                        \
                union {                                                                                \
                    u32x4_t u;                                                                         \
                    bf16x8_t v;                                                                        \
                } w_, a_;                                                                              \
                w_.u = fb[bbuf_][j];                                                                   \
                a_.u = fa[abuf_][i];                                                                   \
                acc[j][(f0_) + i] =                                                                    \
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_.v, a_.v, acc[j][(f0_) + i], 0, 0, 0);   \
            }                                                                                          \
    }
// Order inside a phase of 4 nf MFMAs: its nrd fragment reads go between the first MFMAs, its nvm loads between
// the MFMAs behind them
#define D16_MIX(nf_, nrd_, nvm_)                                                        \
    _Pragma("unroll") for (int g_ = 0; g_ < (nrd_); ++g_) {                             \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, 4 * (nf_) > (nrd_) + 2 ? 4 * (nf_) / ((nrd_) + 2) : 1, 0); \
        __builtin_amdgcn_sched_group_barrier(SG_DS_RD, 1, 0);                           \
    }                                                                                   \
    _Pragma("unroll") for (int g_ = 0; g_ < (nvm_); ++g_) {                             \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);                            \
        __builtin_amdgcn_sched_group_barrier(SG_VMEM, 1, 0);                            \
    }
// phase 3: a fragment read per MFMA over the first half (K-major weights: their four fragments take two read
// instructions each), a load per two MFMAs over the second
#define D16_MIX_DMA(nf0_, nf1_)                                                         \
    _Pragma("unroll") for (int g_ = 0; g_ < 4; ++g_) {                                  \
        __builtin_amdgcn_sched_group_barrier(SG_DS_RD, BKM ? 2 : 1, 0);                 \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);                            \
    }                                                                                   \
    _Pragma("unroll") for (int g_ = 0; g_ < (nf0_); ++g_) {                             \
        __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RA, 0);                          \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);                            \
    }                                                                                   \
    _Pragma("unroll") for (int g_ = 0; g_ < 4; ++g_) {                                  \
        __builtin_amdgcn_sched_group_barrier(SG_VMEM, 1, 0);                            \
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, (nf1_) == 4 ? 2 : 1, 0);          \
    }
// STG: weight stage of slab kt (compile time); s_cur / s_nxt: offsets in the ring of three of slabs kt, kt+1
// (the third stage takes slab kt+2).  Slabs past the end are clamped to the last one (their loads land in
// stages nobody reads again).
// N0 / N1 (compile time): fragments in the first and the second part of the wave's rows.  A wave none of whose
// rows the expert has (0, 0) keeps its loads and barriers but skips its fragment reads and MFMAs.
#define D16_ISSUE_FAR(j_)                                                               \
    {                                                                                   \
        if (MIDROWS) D16_ISSUE_B1(ka_, s_far, j_);                                        \
        else D16_ISSUE_A1(ka_, s_far, j_);                                              \
    }
#define D16_ITER(kt_, STG, N0, N1)                                                      \
    {                                                                                   \
        const int s_far = 3 * A_STAGE - s_cur - s_nxt;                                  \
        const int ca_ = MIDROWS ? STG * A_STAGE : s_cur, na_ = MIDROWS ? (STG ^ 1) * A_STAGE : s_nxt; \
        const int cb_ = MIDROWS ? s_cur : STG * B_STAGE, nb_ = MIDROWS ? s_nxt : (STG ^ 1) * B_STAGE; \
        __builtin_amdgcn_s_setprio(0);                                                  \
        const int kr_ = min((kt_) + 2, nk - 1) + k0, ka_ = kr_ < nk ? kr_ : kr_ - nk;   \
        if (N1) D16_READ_A(ca_, 0, N0, N1, 1);                                       \
        D16_ISSUE_FAR(0);                                                                 \
        if (N0) {                                                                       \
            D16_READ_B(cb_, 1, 0, 1);                                                   \
            D16_READ_B(cb_, 1, 1, 1);                                                   \
            D16_MMA(0, 0, 0, N0);                                                       \
            D16_MIX(N0, N1 * RA + RB2, 1);                                                   \
        }                                                                               \
        PL_FENCE();                                                                     \
        D16_ISSUE_FAR(1);                                                                 \
        if (N0) {                                                                       \
            D16_READ_A(ca_, 1, 0, N0, 0);                                            \
            D16_READ_B(cb_, 1, 2, 1);                                                   \
            D16_READ_B(cb_, 1, 3, 1);                                                   \
        }                                                                               \
        if (N1) {                                                                       \
            D16_MMA(0, 1, N0, N1);                                                      \
            D16_MIX(N1, N0 * RA + RB2, 1);                                                   \
        }                                                                               \
        PL_FENCE();                                                                     \
        D16_ISSUE_FAR(2);                                                                 \
        D16_ISSUE_FAR(3);                                                                 \
        if (N1) D16_READ_A(ca_, 1, N0, N1, 1);                                       \
        if (N0) {                                                                       \
            D16_MMA(1, 0, 0, N0);                                                       \
            D16_MIX(N0, N1 ? N1 * RA : 1, 2);                                                \
        }                                                                               \
        PL_FENCE();                                                                     \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NIA) : "memory"); \
        __builtin_amdgcn_s_setprio(2);                                                  \
        PL_FENCE();                                                                     \
        if (N0) {                                                                       \
            D16_READ_B(nb_, 0, 0, 0);                                               \
            D16_READ_A(na_, 0, 0, N0, 0);                                            \
            D16_READ_B(nb_, 0, 1, 0);                                               \
            D16_READ_B(nb_, 0, 2, 0);                                               \
            D16_READ_B(nb_, 0, 3, 0);                                               \
        }                                                                               \
        if (MIDROWS) D16_ISSUE_A(ka_, STG * A_STAGE)                                       \
        else D16_ISSUE_B(ka_, STG * B_STAGE)                                            \
        if (N1) {                                                                       \
            D16_MMA(1, 1, N0, N1);                                                      \
            D16_MIX_DMA(N0, N1);                                                        \
        }                                                                               \
        PL_FENCE();                                                                     \
        s_cur = s_nxt;                                                                  \
        s_nxt = s_nxt == 2 * A_STAGE ? 0 : s_nxt + A_STAGE;                             \
    }
#define D16_LOOP(N0, N1)                                                                \
    {                                                                                   \
        int kt = 0;                                                                     \
        if (N0) {                                                                       \
            D16_READ_A(0, 0, 0, N0, 0);                                                 \
            _Pragma("unroll") for (int j = 0; j < TN; ++j) D16_READ_B(0, 0, j, 0);      \
        }                                                                               \
        for (; kt + 1 < nk; kt += 2) {                                                  \
            D16_ITER(kt, 0, N0, N1);                                                    \
            D16_ITER(kt + 1, 1, N0, N1);                                                \
        }                                                                               \
        if (kt < nk) D16_ITER(kt, 0, N0, N1);                                           \
    }

    // first two slabs
    const int k0 = ONCE && SWIGLU ? (tc.e / p.sm * ((p.n_tiles + p.sn - 1) / p.sn) + tc.nt / p.sn) % kNumXcd * nk / kNumXcd : 0;
    const int k1 = k0 + 1 < nk ? k0 + 1 : nk > 1 ? 0 : k0;
    D16_ISSUE_B(k0, 0);
    D16_ISSUE_B(k1, B_STAGE);
#pragma unroll
    for (int j = 0; j < NIA && !AKM; ++j) {
        const int64_t src = gather ? (int64_t)(a_idx[j] / p.a_row_div) : (int64_t)a_idx[j];
        ao[j] = (unsigned)(src * p.lda * ES + dchunk * 16);
    }
    D16_ISSUE_A(k0, 0);
    D16_ISSUE_A(k1, A_STAGE);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NIA) : "memory");
    int s_cur = 0, s_nxt = A_STAGE;
    // rows of the expert in this wave's share of the tile (wave-uniform)
    const int wave_row = tile_row + wm * share0;
    int wave_rows = count - wave_row;
    if constexpr (MIDROWS) {
        wave_rows = wave_rows < frags * 16 ? wave_rows : frags * 16;
        switch (frags) {
            case 8: D16_LOOP(4, 4) break;
            case 7: D16_LOOP(4, 3) break;
            case 6: D16_LOOP(3, 3) break;
            case 5: D16_LOOP(3, 2) break;
            case 4: D16_LOOP(2, 2) break;
            case 3: D16_LOOP(2, 1) break;
            default: D16_LOOP(1, 1) break;
        }
    } else if (wave_rows > 64) {
        D16_LOOP(4, 4)
    } else if (wave_rows > 0) {
        D16_LOOP(4, 0)
    } else {
        D16_LOOP(0, 0)
    }
    __builtin_amdgcn_s_setprio(0);
    // the clamped loads of the last slabs may still be in flight; the epilogue reuses LDS
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#undef D16_LOOP
#undef D16_LOAD
#undef D16_ISSUE_A
#undef D16_ISSUE_A1
#undef D16_ISSUE_B
#undef D16_ISSUE_B1
#undef D16_ISSUE_FAR
#undef D16_B_ROW
#undef D16_READ_A
#undef D16_READ_B
#undef D16_MMA
#undef D16_MIX
#undef D16_MIX_DMA
#undef D16_ITER

    {
        typedef AccView16<TM, TN, SWIGLU> View;
        constexpr int WSTAGE = epilogue_wstage_bytes<TO, View, DSILU>();
        const int ncol0 = SWIGLU ? tc.nt * HALF + wn * (BN / WN / 2) : tc.nt * BN + wn * (BN / WN);
        if constexpr (SAVEGU || DSILU) {
            constexpr int TSTAGE = SAVEGU ? kTransStageH : kTransStageD;
            static_assert(NW * (WSTAGE + TSTAGE) <= (3 * BM + 2 * BN) * 128, "epilogue staging exceeds the tile's LDS");
            TO* tout = static_cast<TO*>(p.t_out);
            const int64_t tcol = tout ? (int64_t)p.t_col0[tc.e] + wave_row : 0;
            epilogue_view<TO, View, SWIGLU, SAVEGU, DSILU>(View{acc}, smem + wave * WSTAGE, static_cast<TO*>(p.out), p.ldo,
                                                           (int64_t)row0 + wave_row, wave_rows, ncol0, p.N_out, lane,
                                                           static_cast<TO*>(p.gu_out), p.ld_gu, p.up_offset, tout,
                                                           p.ld_t, tcol, smem + NW * WSTAGE + wave * TSTAGE);
        } else {
            TO* const out = static_cast<TO*>(p.out) + (SLICED ? (int64_t)split * p.part_stride : 0);
            epilogue_view<TO, View, SWIGLU, SAVEGU, DSILU>(View{acc}, smem + wave * WSTAGE, out, p.ldo,
                                                           (int64_t)row0 + wave_row, wave_rows, ncol0, p.N_out, lane,
                                                           static_cast<TO*>(p.gu_out), p.ld_gu, p.up_offset);
        }
    }
#endif
}

template <typename TO, int SM, int SN, bool SWIGLU, bool SAVEGU = false, bool DSILU = false, bool BKM = false,
          bool MIDROWS = false, bool SLICED = false, bool AKM = false, bool ONCE = false>
__global__ __launch_bounds__(512) void grouped_gemm_dma16_kernel(GroupedArgs p) {
    // The body is a function of its own for one reason: a __restrict__ parameter that it reads through gives every
    // other memory access in it (the transposing LDS reads among them) "does not alias that parameter" metadata once
    // it is inlined here, and the compiler's wait insertion takes an LDS read that carries alias metadata but no
    // scope of a direct-to-LDS load as independent of the loads in flight.  Without it every ds_read_b64_tr_b16 of
    // the K-major variant is preceded by s_waitcnt vmcnt(0), i.e. waits for all of the slab loads just issued (the
    // plain 16-byte fragment reads carry type-based alias metadata and never had that wait): 27-37 % slower.
    extern __shared__ __align__(16) unsigned char smem_k[];
    grouped_gemm_dma16_body<TO, SM, SN, SWIGLU, SAVEGU, DSILU, BKM, MIDROWS, SLICED, AKM, ONCE>(p, smem_k, p.row_count);
}

#undef PL_STORE
#undef PL_READ
#undef PL_MMA
#undef PL_FENCE
#undef PL_MIX_READS

}  // namespace ats

#include "grouped_gemm_short.hpp"
#include "grouped_gemm_band.hpp"

namespace ats {

// LDS of the direct-to-LDS kernel: three activation stages and two weight stages of unpadded 128-byte rows.
constexpr size_t dma_lds_bytes(int BM, int BN) { return (size_t)(3 * BM + 2 * BN) * 128; }

// Rows per group on average below which the 16 x 16 x 32 kernel runs in its MIDROWS form (measured there).
constexpr int64_t kMidRowsMaxAvg = 768;
// Rows per group on average up to which hardly any group exceeds a tile's 256 rows where the groups are about equal.
constexpr int64_t kOnceMaxAvgRows = 224;
// The ONCE instance.  Only the mean of the groups is known here.  With sizes that fall as rank^-1.5 the larger ones take two or three tiles
// and load their weights non-temporally in each, and it still gains where the weights are large: 110 .. 222 rows on average, gate/up 8 x
// [28672, 4096] 0.96 .. 1.00 of the time, 64 x [2816, 2048] 0.94 .. 0.97, 12 x [8192, 3072] 1.00 .. 1.03, sliced down 8 x [4096, 14336]
// 0.91 .. 0.95, 16 x [2048, 5632] 0.95 .. 0.98 (equal chances: 0.90 .. 0.98, 0.80 .. 0.94, 0.93 .. 0.97, 0.86 .. 0.95, 0.84 .. 0.94).  Sliced
// products of less than a last-level cache of weights (256 MB) gain nothing and lose where the sizes differ: 8 x [1024, 2816] 31.3 -> 35.1
// us, equal chances 41.3 -> 41.5.  Small gate/up products by themselves are even (8 x [5632, 1024] 31.0 -> 30.5, 45.0 -> 46.4), but leave the
// cache to the down projection behind them: the layer 82 -> 76 us, 98 -> 95.  (A choice per group inside the kernel, as the band tiles make
// it, costs more than it saves: with both bodies, or with a branch at the loads, registers spill and skewed groups take 1.1 .. 1.9 times as
// long.)
static bool once_weights(int64_t max_rows, int E) { return E > 1 && max_rows / E <= kOnceMaxAvgRows; }
static bool once_slices(int64_t max_rows, int E, int N, int K) { return once_weights(max_rows, E) && (int64_t)E * N * K >= (int64_t)1 << 27; }
static bool mid_rows(int64_t max_rows, int E) { return max_rows / (E > 0 ? E : 1) < kMidRowsMaxAvg; }
// Tiles of the busiest CU.  Supertile S runs on XCD S % 8; the last band of rows and the last one of columns hold fewer than 32 tiles
// (18 x 43 tiles of 256 rows: 33 supertiles, five for XCD 0, of which one has eight tiles and the others leave it four rounds).
static int64_t busiest_cu(int64_t m_tiles, int n_tiles, int sm, int sn) {
    const int64_t bands = (m_tiles + sm - 1) / sm, super = bands * ((n_tiles + sn - 1) / sn);
    if (super > 256) return (super + kNumXcd - 1) / kNumXcd;
    int64_t tiles[kNumXcd] = {}, most = 0;
    for (int64_t i = 0; i < super; ++i) {
        const int64_t rows = m_tiles - i % bands * sm, cols = n_tiles - i / bands * sn;
        tiles[i % kNumXcd] += (rows < sm ? rows : sm) * (cols < sn ? cols : sn);
    }
    for (int64_t t : tiles) most = t > most ? t : most;
    return (most + kSuperBlocks - 1) / kSuperBlocks;
}

// Tile height of a bfloat16 launch with one group (its row count is exact) on the 256-row tile, 0 for the full 256 rows.  An XCD takes whole
// supertiles of 32 tiles and its 32 CUs hold one tile each, so a launch lasts as many rounds as there are supertiles per XCD,
// and lower tiles pay where they turn a round that is mostly empty into work for all CUs (4524 x [11008, 2048]: 240 rows in four
// rounds 174 us, 144 rows in six 215).  Microseconds per 64-element slab by height: medians over 415
// launches.
// Rows x [N, K], 256-row tiles -> heights in steps of 32 -> in steps of 16: 5331 x [4096, 4096] 188 -> 143 -> 134 us, x
// [6144, 4096] 248 -> 207 -> 200, 4200 x [4096, 4096] 123 -> 116, 10000 x [6144, 4096] 369 -> 346, 5331 x [3072, 2048] 67 -> 62,
// 3000 x [4096, 4096] 95 -> 76 -> 74, 1500 x [4096, 4096] 78 -> 58 -> 56, 1000 x [6144, 4096] 93 -> 57 -> 56; 2048 x [6144, 4096]
// stays (92; 128 rows 113).  Weights stored [K][N] take the same heights: 1000 x [4096, 4096] 90 -> 55, 300 x 55 -> 49, 5331 x
// 176 -> 136, x [6144, 4096] 238 -> 202, 2048 x [2048, 2048] 50 -> 32.  Sums over K are in the same order.
static int dense_tile_rows(int64_t rows, int n_tiles, int k_slabs, int sm, int sn, float* time = nullptr) {
    float best = 0.f;
    int best_rows = 0;
    constexpr float kPerSlab[] = {0.75f, 0.86f, 0.94f, 1.00f, 1.07f, 1.15f, 1.23f, 1.28f, 1.35f};     // 128, 144, .. 256 rows
    for (int h = 256; h >= 128; h -= 16) {
        const int64_t m_tiles = (rows + h - 1) / h;
        const int64_t height = ((rows + m_tiles - 1) / m_tiles + 15) / 16 * 16;     // tiles of a group have one height
        const float per_slab = kPerSlab[height > 128 ? (height - 128) / 16 : 0];
        const float t = (float)busiest_cu(m_tiles, n_tiles, sm, sn) * (k_slabs * per_slab + 7.f);
        if (h == 256 || t < 0.97f * best) {
            best = t;
            best_rows = h == 256 ? 0 : h;
        }
    }
    if (time) *time = best;
    return best_rows;
}

template <typename T, typename TO, int BM, int BN, int WM, int WN, int SM, int SN, bool SWIGLU, bool DMA = false>
static int launch_cfg(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    GroupedArgs p = p0;
    constexpr int n_per_tile = SWIGLU ? BN / 2 : BN;
    p.n_tiles = (p.N_out + n_per_tile - 1) / n_per_tile;
    // register-staged kernels: two padded stages; direct-to-LDS kernel: three activation + two weight stages
    constexpr size_t smem_staged = 2 * (size_t)(BM + BN) * kRowPitch;
    constexpr size_t smem = DMA && dma_lds_bytes(BM, BN) > smem_staged ? dma_lds_bytes(BM, BN) : smem_staged;
    constexpr int BK = 128 / (int)sizeof(T);
    // slices of K: the 32 and 64-row tiles, whose only instance is the sliced one of the register-staged kernel
    constexpr bool kSliced = !DMA && !SWIGLU && (BM == 32 || BM == 64);
    // the L2 warm-up touches pay where blocks share operand panels; the weight-streaming tiles share nothing
    constexpr bool kWarm = BM > 64;
    auto kern_pipe = grouped_gemm_pipelined_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU, kWarm, kSliced>;
    auto kern_general = [] {
        if constexpr (kSliced) return grouped_gemm_pipelined_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU, kWarm, true>;
        else return grouped_gemm_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU>;
    }();
    auto kern_dma = [] {
        if constexpr (DMA && std::is_same<T, bf16_t>::value) {
            static_assert(BM == 256 && BN == 256 && WM == 2 && WN == 4, "the 16 x 16 x 32 kernel is the 256 x 256 tile");
            return grouped_gemm_dma16_kernel<TO, SM, SN, SWIGLU>;
        } else if constexpr (DMA) return grouped_gemm_dma_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU>;
        else return grouped_gemm_pipelined_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU, kWarm, kSliced>;
    }();
    auto kern_mid = [] {       // groups of a few hundred rows
        if constexpr (DMA && std::is_same<T, bf16_t>::value) return grouped_gemm_dma16_kernel<TO, SM, SN, SWIGLU, false, false, false, true>;
        else if constexpr (DMA) return grouped_gemm_dma_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU>;
        else return grouped_gemm_pipelined_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU, kWarm, kSliced>;
    }();
    auto kern_once = [] {      // one tile per group
        if constexpr (DMA && SWIGLU && std::is_same<T, bf16_t>::value)
            return grouped_gemm_dma16_kernel<TO, SM, SN, true, false, false, false, true, false, false, true>;
        else if constexpr (DMA && std::is_same<T, bf16_t>::value) return grouped_gemm_dma16_kernel<TO, SM, SN, SWIGLU, false, false, false, true>;
        else if constexpr (DMA) return grouped_gemm_dma_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU>;
        else return grouped_gemm_pipelined_kernel<T, TO, BM, BN, WM, WN, SM, SN, SWIGLU, kWarm, kSliced>;
    }();
    if (smem > 64 * 1024) {
        static LdsReservation reserved;      // one per tile configuration (this function is a template)
        hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern_general),
                                              reinterpret_cast<const void*>(kern_pipe),
                                              reinterpret_cast<const void*>(kern_dma),
                                              reinterpret_cast<const void*>(kern_mid),
                                              reinterpret_cast<const void*>(kern_once)}, (int)smem);
        if (e != hipSuccess) {
            set_error("grouped GEMM: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
            return ATS_ERR_LAUNCH;
        }
    }
    const int splits = p.k_splits > 1 ? p.k_splits : 1;
    if ((splits > 1) != kSliced || (kSliced && (p.k_count || p.K % splits != 0 || (p.K / splits) % BK != 0))) {
        set_error("grouped GEMM: %d slices of K=%d are not available for this tile configuration", splits, p.K);
        return ATS_ERR_UNSUPPORTED;
    }
    // the prefill / mid-size tiles take the supertile shape that leaves the fewest n-slots unused; the
    // weight-streaming tiles keep theirs (one m-tile per group, 32 n-tiles side by side)
    p.sm = SM;
    p.sn = SN;
    if (SM == 4 && SN == 8) pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = max_rows / (p.E > 0 ? p.E : 1) >= kAlignedBandsMinAvgRows ? 1 : 0;
    // the direct-to-LDS kernel addresses its operands with 32-bit lane offsets
    const bool dma_ok = DMA && p.K % BK == 0 && p.a_extent_bytes != 0 && p.b_extent_bytes != 0;
    p.tile_rows = 0;
    if (dma_ok && std::is_same<T, bf16_t>::value && p.E == 1)
        p.tile_rows = dense_tile_rows(max_rows, p.n_tiles, p.K / BK, p.sm, p.sn);
    const int64_t blocks = grid_blocks(max_rows * splits, p.E * splits, p.tile_rows ? p.tile_rows : BM, p.n_tiles, p.sm, p.sn,
                                       p.aligned_bands != 0);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    const bool once = once_weights(max_rows, p.E);
    auto kern = dma_ok ? (once ? kern_once : p.tile_rows || mid_rows(max_rows, p.E) ? kern_mid : kern_dma) : (p.K % BK == 0) ? kern_pipe : kern_general;
    const size_t smem_launch = (!dma_ok && p.K % BK == 0) ? smem_staged : smem;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(WM * WN * 64), smem_launch, s, p);
    return ATS_OK;
}

// K in slices over workgroups on the direct-to-LDS tile, groups of 21 .. 256 rows: float32 partial results.  A down projection
// of few experts has half a round of these tiles or less (8 x [4096, 14336]: 128), and a CU takes 1.2-1.4 us per slab of
// K whatever the other half of the chip does; two slices make it a full round: 200 rows per expert 314 -> 165 us.  The 32
// and 64-row sliced tiles it replaces for several groups read every weight once per 64 rows (200 rows: 517 us).
template <bool BKM = false>
static int launch_mid_sliced(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + 255) / 256;
    constexpr size_t smem = dma_lds_bytes(256, 256);
    auto kern_many = grouped_gemm_dma16_kernel<float, 4, 8, false, false, false, BKM, true, true>;
    auto kern_once = grouped_gemm_dma16_kernel<float, 4, 8, false, false, false, BKM, true, true, false, !BKM>;
    auto kern = once_slices(max_rows, p.E, p.N_out, p.K) ? kern_once : kern_many;
    static LdsReservation reserved;
    hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern_many), reinterpret_cast<const void*>(kern_once)}, (int)smem);
    if (e != hipSuccess) {
        set_error("grouped GEMM: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
        return ATS_ERR_LAUNCH;
    }
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = 0;
    p.tile_rows = 0;
    const int64_t blocks = grid_blocks(max_rows * p.k_splits, p.E * p.k_splits, 256, p.n_tiles, p.sm, p.sn, false);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(512), smem, s, p);
    return ATS_OK;
}

// Time of a launch on one tile configuration, in microseconds, from the number of tiles that the busiest CU gets:
// every tile costs per_slab for each 128-byte slab of K (with the CU's other resident tiles running beside it) and
// per_tile for its set-up and epilogue.  min_tiles: below that many tiles per CU nothing hides the latency of a slab,
// so fewer tiles are not faster.
struct TileCost {
    int rows, cols;
    float per_slab, per_tile;
    int min_tiles;
};
// spread: groups vary around their mean, so those of a mean just below a multiple of the tile height need one tile more; counted as
// rows / spread more of them.
static float tile_time(const TileCost& c, int64_t max_rows, int E, int n_cols, int k_slabs, int spread = 0) {
    const int64_t rows = spread && E > 1 ? max_rows + max_rows / spread : max_rows;
    const int64_t avg = (rows + E - 1) / E;
    const int64_t tiles = (int64_t)E * ((avg + c.rows - 1) / c.rows) * ((n_cols + c.cols - 1) / c.cols);
    const int64_t per_cu = (tiles + 255) / 256;
    return (float)(per_cu > c.min_tiles ? per_cu : c.min_tiles) * (k_slabs * c.per_slab + c.per_tile);
}

// Tile configuration by the size of the launch: the one with the least estimated time.  The constants were measured on
// MI355X, one launch of each configuration over [33 .. 5331] x [1024 .. 6144] x [64 .. 4096] products and over 8 and
// 64 groups of 40 .. 384 rows.  What the rule decides between, in microseconds:
//   in-block slices of K, 32 rows | 64 rows | 128 rows, register-staged | 256 rows, direct to LDS
//   bfloat16  128 x 4096 x 4096    17 |  23 |  48 |  44      float32   512 x  512 x  512     9 |   17 |  62 | 120
//             300 x 4096 x 4096    37 |  34 |  61 |  71                512 x 2816 x  512    25 |   29 |  67 | 122
//            1024 x 4096 x 4096    98 |  72 |  68 |  94               1000 x 1000 x 1000    33 |   29 | 157 | 262
//            2048 x 4096 x 4096   192 | 130 |  69 |  97               2048 x 2048 x 2048   219 |  180 | 246 | 467
//            5331 x 4096 x 4096   472 | 310 | 197 | 184               4096 x 4096 x 4096  1498 | 1193 | 944 | 937
//   gate/up, 8 groups of 160, I 14336   942 | 762 | 572 | 408
//   float32 in 2 x 2 tiles of 32 rows without slices of K: 2048 x 512 x 512 19 (128 rows: 67, 256 rows: 122)
// Two bounds on the choice keep results independent of the route that a training step takes: bfloat16 groups of more
// than 192 rows always run on the 16 x 16 x 32 kernel and float32 groups of more than 256 rows are not sliced along K,
// because the fused training launches and the K-major products, which start at those sizes, accumulate in that order
// (their results equal those of the separate launches bit for bit).  The gate/up product with its activation, which training does not
// run (it rounds the pre-activations that it keeps), is outside of that: up to kOnceMaxAvgRows it begins K elsewhere.
enum class GroupTile { kSmall32, kSmall64, kSeq, kMid, kBig };      // kSeq: 64 rows, all of K in a wave
template <bool kBf16, bool SWIGLU>
static GroupTile pick_group_tile(int64_t max_rows, int E, int N, int nk) {
    const int64_t avg = max_rows / E;
    // (columns: output columns per tile, half of the weight rows with the SwiGLU epilogue)
    constexpr TileCost kSmall32 = kBf16 ? TileCost{32, 32, SWIGLU ? 0.165f : 0.093f, 1.f, SWIGLU ? 1 : 2}
                                        : TileCost{32, 32, SWIGLU ? 0.40f : 0.18f, 1.5f, 1};
    constexpr TileCost kSmall64 = kBf16 ? TileCost{64, SWIGLU ? 32 : 64, 0.245f, 1.5f, 1}
                                        : TileCost{64, SWIGLU ? 32 : 64, 0.58f, 3.f, 1};
    constexpr TileCost kMid = kBf16 ? TileCost{128, SWIGLU ? 64 : 256, SWIGLU ? 0.58f : 1.05f, 5.f, 1}
                                    : TileCost{128, SWIGLU ? 64 : 256, SWIGLU ? 2.0f : 3.65f, 5.f, 1};
    // A fifth where many groups make it likely that one of them is that much larger (64 experts of 108 rows on average, 81-140: gate/up
    // 182 us in 128-row tiles, 161 in 256-row ones; of 94 rows 167 both), a tenth for a few (4 experts of 110 rows, [16384, 2048]: 67.5
    // us, with a fifth 74) and in float32, whose tiles of 128 rows lose less than the taller ones (2 x 226 rows, [8192, 1024]: 66 us, with a
    // fifth 88; 32 x 225 rows, [1536, 1024]: 188, 241; 4 x 331 rows, [16384, 2048]: 734, 944).
    const int spread = kBf16 && E >= 8 ? 5 : 10;
    const float mid = tile_time(kMid, max_rows, E, N, nk, spread);
    // (the 16 x 16 x 32 kernel computes only the 16-row fragments that a tile has; up to 192 rows its loads bound a slab)
    const float big = tile_time(TileCost{256, SWIGLU ? 128 : 256, kBf16 ? (avg <= 192 ? 1.3f : 1.45f) : 7.3f, 7.f, 1},
                                max_rows, E, N, nk, spread);
    const float least_large = mid < big ? mid : big;
    // (two full rounds of 256-row tiles: nothing is idle, and groups of unequal size fit them better; 8 experts with 20-45
    // rows each, gate/up [28672, 4096]: 343 us against 372 in 32-row tiles)
    const int64_t big_tiles = (int64_t)E * ((avg + 255) / 256) * ((N + (SWIGLU ? 127 : 255)) / (SWIGLU ? 128 : 256));
    if (big_tiles < 512) {
        if (avg <= (kBf16 ? 192 : 256)) {
            const float small32 = tile_time(kSmall32, max_rows, E, N, nk);
            // (a long K streams the weights from HBM: 8 groups x 128 rows, [4096, 14336]: 328 us against 258 in 128-row tiles)
            TileCost c64 = kSmall64;
            if (kBf16 && nk >= 128) c64.per_slab = 0.3f;
            const float small64 = tile_time(c64, max_rows, E, N, nk);
            if (small32 < least_large && small32 <= small64) return GroupTile::kSmall32;
            if (small64 < least_large) return GroupTile::kSmall64;
        } else if constexpr (!kBf16) {
            constexpr TileCost kSeq = TileCost{64, 64, SWIGLU ? 1.4f : 0.74f, 3.f, 1};
            if (tile_time(kSeq, max_rows, E, N, nk) < least_large) return GroupTile::kSeq;
        }
    }
    return mid < big && !(kBf16 && avg > 192) ? GroupTile::kMid : GroupTile::kBig;
}

// up to 32 rows per expert against a long K, for callers that do not cut K (8 experts x 32 rows, [4096, 14336], with
// the combine behind it: 178 us, 21 rows 165; two slices of K over workgroups 165 and 163; the launch in 256-row tiles
// 264)
static bool streams_long_k(int64_t avg, int pieces, int N) { return avg <= 32 && pieces >= 64 && N >= 32; }

// A bfloat16 projection of E experts with 21 .. 256 rows each and 32 MB of weights or more, plain or in s slices of K, with the
// combine behind it, in microseconds: a workgroup's chain of slabs and the weights from HBM, which overlap in part (hence the
// root of the squares), the start, and the partial results written and read.  What the chain depends on is how the workgroups
// fill the chip: two of the 64-row tiles share a CU, a third is a second round; the 256-column tiles come in supertiles of 32
// that belong to one XCD each, so that ten tiles of a row band leave some XCDs a second round and others idle.  Fitted to 8071
// points, 2 .. 64 experts, 512 .. 8192 columns, K from 1024 to 16384, uneven groups, weights from HBM: within 7 % (256 columns)
// to 11 % (slices on the small tiles) of the times, root mean square.
struct SliceEstimate {
    int E, N, K;
    int64_t max_rows;
    float avg, slabs, weights, partials;      // megabytes of the weights and of one slice's results, written and read
    SliceEstimate(int E_, int64_t max_rows_, int N_, int K_) : E(E_), N(N_), K(K_), max_rows(max_rows_) {
        avg = (float)max_rows / E;
        slabs = K / 64.f;
        weights = (float)E * N * K * 2e-6f;
        partials = (float)max_rows * N * 8e-6f;
    }
    // Tiles of bm rows per group, on average over groups whose sizes vary by their square root.
    float row_tiles(float bm) const {
        const float t = ceilf(avg / bm), w = 1.7f / sqrtf(avg);
        return t + 1.f / (1.f + expf(w * (t * bm - avg))) - (t > 1.f ? 1.f / (1.f + expf(w * (avg - (t - 1.f) * bm))) : 0.f);
    }
    static float join(float a, float b) { return sqrtf(a * a + b * b); }
    // bm rows x 256 columns, one to a CU; pitch: rows of 8 KB or a multiple of it ask few of the memory's channels at a time
    struct Tall { float bm, slab, slab_row, tile, rate, start, parts, pitch; };
    float tall(const Tall& c, int s, float* rounds_out = nullptr) const {
        const int n_tiles = (N + 255) / 256;
        int sm, sn;
        pick_supertile(n_tiles, &sm, &sn);
        const float m = s * roundf(E * row_tiles(c.bm)), super = ceilf(m / sm) * ((n_tiles + sn - 1) / sn);
        const float rounds = fmaxf(1.f, ceilf(ceilf(super / kNumXcd) * (m * n_tiles / (super * kSuperBlocks)) - 0.02f));
        if (rounds_out) *rounds_out = rounds;
        const float chain = rounds * (slabs / s * (c.slab + c.slab_row * fminf(avg, c.bm)) + c.tile);
        const float load = weights / c.rate * sqrtf(sqrtf(kNumXcd / fminf(super, kNumXcd))) * (K % 4096 == 0 ? 1.f + c.pitch : 1.f);
        return c.start + join(chain, load) + partials * s / c.parts;
    }
    float large(int s, float* rounds = nullptr) const { return tall(Tall{256.f, 0.75f, 0.0016f, 7.7f, 6.5f, 5.1f, 5.7f, 0.11f}, s, rounds); }
    // Slices on it against the band tiles.  Fitted before the ONCE instance, which takes 4 .. 14 % less where one round of tiles fills the
    // chip and rows are no multiple of 8 KB: 8 x [4096, 14336] of 48 .. 72 rows in two slices 158-161 us, on the band tiles 164-172.  Where sizes
    // fall as rank^-1.5 its taller tiles hold the largest group (two fifths of all rows) up to 600 rows in all: 166-176 for 182-193.
    bool large_beats_band(int s) const {
        float rounds;
        const float time = large(s, &rounds) + 2.f;
        return s > 1 && avg <= 72.f && max_rows <= 600 && once_slices(max_rows, E, N, K) && K / s >= 512 && rounds == 1.f && K % 4096 != 0 &&
               0.93f * time < fminf(small(s), band(s));
    }
    // 32 or 64 rows x 128 columns, slices of K over workgroups; a row band is launched as whole supertiles of 32 columns' tiles, and
    // the workgroups without a tile cost a microsecond per round
    float small(int s) const {
        const bool few = max_rows / E <= 32;
        const float n = slabs / s, bands = E * s * row_tiles(few ? 32.f : 64.f), n_tiles = (N + 127) / 128;
        const float tiles = bands * n_tiles / 256.f, pc = fmaxf(1.f, tiles);
        const float empty = bands * (float)((N + 4095) / 4096) * 32.f / 256.f - tiles;
        if (few) return 7.6f + n * (0.476f + 0.207f * pc + (pc > 3.1f ? 0.381f : 0.f)) + 0.476f * pc + 0.913f * empty + weights / 11.2f;
        const float chain = n * (0.325f + 0.377f * pc + (pc > 2.12f ? 0.367f : 0.f)) + 0.077f * pc + 1.02f * empty;
        return 8.6f + powf(powf(chain, 1.36f) + powf(weights / 9.7f, 1.36f), 1.f / 1.36f) + partials * s / 13.5f;
    }
    // The band tiles, where band_groups takes them: one tile to a CU or several, whose slabs then follow one another.  Fitted to 791 points
    // of groups with equal chances, 2 .. 64 experts of 21 .. 100 rows on average, [768 .. 5120, 1408 .. 14336] weights, within 5 % (18 % at
    // most).  Where plain tiles just fill the CUs once, sizes that differ more give some of them a second one: with sizes that fall as
    // rank^-1.5, 8 x [4096, 14336] of 50 rows take 226 us plain and 193 in two slices, with equal chances 154 and 164.  Hence 11 % on such
    // launches: what is chosen is 1.4 % slower than the fastest of every route with equal chances and 3.5 % with such sizes (by the
    // estimates of the tiles that ran there before 6 and 7 %, without the 11 % 0.8 and 6).
    float band(int s) const {
        const float used = E * (1.f - expf(-avg)) * (1.f + 1.f / (1.f + expf(1.7f / sqrtf(avg) * (128.f - avg))));
        const float pc = used * ((N + kBandCols - 1) / kBandCols) * s / 256.f;
        const bool alone = pc <= 1.02f;
        const float slab = alone ? 0.481f + 0.0022f * avg : (0.431f + 0.0021f * avg) * (0.07f * pc + 0.93f * ceilf(pc - 0.02f));
        const float chain = slabs / s * slab, load = weights / (alone ? 6.9f : 6.24f);
        const float time = 8.3f + powf(powf(chain, 5.f) + powf(load, 5.f), 0.2f) + (s > 1 ? 2.6f + partials * s / 5.43f : partials / 6.46f);
        return s == 1 && alone && pc > 0.8f ? 1.11f * time : time;
    }
    float plain() const {
        if (streams_long_k(max_rows / E, K * 2 / 256, N)) return 8.65f + join(slabs * 0.172f, weights / 5.3f);
        switch (pick_group_tile<true, false>(max_rows, E, N, (K + 63) / 64)) {
            case GroupTile::kSmall32: return 8.06f + join(slabs * 0.164f, weights * (1.f + 0.497f * (row_tiles(32.f) - 1.f)) / 5.24f);
            case GroupTile::kSmall64: {
                const float r = row_tiles(64.f), pc = E * r * ((N + 63) / 64) / 256.f;
                return 8.63f + join(slabs * (0.271f + (pc > 2.12f ? 0.318f : 0.f)), weights * (1.f + 0.396f * (r - 1.f)) / 5.28f) + partials / 4.65f;
            }
            case GroupTile::kMid: return tall(Tall{128.f, 0.897f, 0.f, 2.5f, 6.83f, 2.f, 4.7f, 0.108f}, 1);
            default: return tall(Tall{256.f, 0.656f, 0.0018f, 8.f, 5.8f, 2.6f, 8.5f, 0.064f}, 1);
        }
    }
    // What the plain launch and the slices on the small tiles have to exceed before the large one is taken: the estimates are off by a
    // few microseconds and, where groups come close to a second row tile, by more.
    float large_with_margin(int s) const { return large(s) * (avg <= 64.f ? 1.f : avg <= 208.f ? 1.03f : 1.06f) + 2.f; }
};
// Whether slices of K run on the direct-to-LDS tile.  Slices of less than 512 columns, which no rule asks for and nothing was fitted
// to: with tiles for half of the CUs.  Less than 32 MB of weights come from the last-level cache: never.
static bool large_slice_tile(int E, int64_t max_rows, int N, int K, int s) {
    if (K / s < 512) return (int64_t)E * ((N + 255) / 256) * s >= 128;
    if ((int64_t)E * N * K < (1 << 24)) return false;
    const SliceEstimate t(E, max_rows, N, K);
    return t.large_with_margin(s) < t.small(s) || t.large_beats_band(s);
}

// The band tiles (grouped_gemm_band.hpp) for E > 1 groups.  They lose where a group needs a second tile while the first ones fill no
// more than one round of the chip (8 x [4096, 14336] in two slices, unequal groups of 72 rows 189 -> 230 us, of 56 rows 181 -> 164), and
// among many workgroups where most groups do (64 x [2816, 2048], 96 rows each 176 -> 143, 128 rows 169 -> 180); with a few rows per
// group the weight streams' narrower panels leave fewer CUs idle (16 x [2048, 5632], 16 rows in all 44 -> 52, 32 rows 60 -> 53; 64 x
// [2048, 1408], 6 rows 11 -> 14, 18 rows 19 -> 16) and their gate/up launch is the faster one up to about twelve rows per group
// (64 x [2816, 2048], 4 rows each 107 -> 111, 12 rows 114 -> 114, 16 rows 122 -> 115).
static bool band_groups(int E, int64_t max_rows, int n_tiles, int slices, bool swiglu) {
    const int64_t avg = max_rows / E;
    if (avg > ((int64_t)E * n_tiles >= 512 ? 100 : 72)) return false;
    if (swiglu) return avg >= 12 && (int64_t)E * n_tiles >= 256;
    const float used = E * (1.f - expf(-(float)max_rows / E));      // groups that get rows, if these fall at random
    return used * n_tiles * slices >= 200.f;
}
// One group of more than 32 rows x [N, K]: the band tiles' time in microseconds, plain or with s slices of K and their sum, by the
// tiles' most rows h.  A CU takes one slab of a tile in slab1 alone and in slabn as one of several.  Fitted to 1500 launches of 33 .. 1000
// rows x [512 .. 32000, 512 .. 14336], weights from HBM, within 6 % (root mean square; 22 % at most).
static float band_time(int64_t rows, int N, int K, int s, int h) {
    constexpr float slab1[] = {0.44f, 0.55f, 0.67f}, slabn[] = {0.44f, 0.48f, 0.54f};      // up to 64, 96, 128 rows
    const int64_t m_tiles = (rows + h - 1) / h;
    const int f = std::max((int)((rows + m_tiles - 1) / m_tiles + 31) / 32 - 2, 0);
    const float per_cu = (float)(m_tiles * ((N + kBandCols - 1) / kBandCols) * s) / 256.f;
    const float slab = per_cu <= 1.f ? slab1[f] : slabn[f] * 0.5f * (per_cu + ceilf(per_cu));
    const float chain = K / 64.f / s * slab, weights = (float)N * K * 2e-6f / (per_cu <= 1.f ? 5.6f : 6.1f);
    return 3.6f + sqrtf(chain * chain + weights * weights) + (s > 1 ? (float)rows * N * (8 * s - 4) / 4.75e6f + 2.7f : 0.f);
}
static int band_height(int64_t rows, int N, int K, int s) {
    return rows > 64 && band_time(rows, N, K, s, 128) < band_time(rows, N, K, s, 64) ? 128 : 64;
}
// The same rows on the tile that pick_group_tile takes for them: up to 192 rows the register-staged ones, two workgroups of which share a
// CU (the launches above, within 9 %), beyond that the 256-column tile.  What the choice between the two and the slices costs over those
// launches is 0.9 % on average, 18 % at most (with the constants of 109 points of [2048 .. 6144] x [2048, 4096], and small tiles also
// beyond 192 rows, where none run: 5.6 %, 140 %).  Microseconds, band tiles <- other: 200 rows x [512, 512] 6.9 <- 10.5, [1024, 1024] 10.3 <- 15.0,
// 512 x [1024, 4096] 32 <- 56, 100 x [32000, 4096] 67 <- 91; other <- band tiles: 160 x [3072, 1024] 9.0 <- 10.6, 64 x [2048, 2048] 9.5 <- 17.
static float other_dense_time(int64_t rows, int N, int K) {
    const float slabs = K / 64.f, weights = (float)N * K * 2e-6f;
    switch (pick_group_tile<true, false>(rows, 1, N, (K + 63) / 64)) {
        case GroupTile::kSmall32: {
            const float half = (float)((rows + 31) / 32 * ((N + 31) / 32)) / 512.f;
            const float chain = slabs * (0.166f + 0.068f * fminf(half, 1.f)) * ceilf(half);
            return 3.9f + powf(powf(chain, 3.2f) + powf(weights / 2.41f, 3.2f), 1.f / 3.2f);
        }
        case GroupTile::kSmall64: return 4.4f + slabs * 0.318f * ceilf((float)((rows + 63) / 64 * ((N + 63) / 64)) / 512.f) + weights / 6.2f;
        case GroupTile::kMid: return 4.f + weights / 3.f;
        default: break;
    }
    float best;
    int sm, sn;
    const int n_tiles = (N + 255) / 256;
    pick_supertile(n_tiles, &sm, &sn);
    dense_tile_rows(rows, n_tiles, K / 64, sm, sn, &best);
    return 1.1f * best;      // (the heights are held against each other there, not against other kernels: 300 x [12288, 4096] 62 us for 55)
}
static bool band_dense(int64_t rows, int N, int K) {
    return rows > 32 && band_time(rows, N, K, 1, band_height(rows, N, K, 1)) < other_dense_time(rows, N, K);
}

// The kernel of a launch.  Streams: panels of np * 16 weight rows, tiles of mt * 16 activation rows, kw waves along K.
enum class Route { kSlices32, kSlices64, kSlices256, kBandSlices, kBand, kShort, kStream, kSmall32, kSmall64, kSeq, kMid, kBig };
struct GroupedRoute {
    Route kernel;
    int np, mt, kw;
};

template <typename T, typename TO, bool SWIGLU>
static GroupedRoute grouped_route(const GroupedArgs& p, int64_t max_rows) {
    constexpr bool kBf16 = std::is_same<T, bf16_t>::value;
    constexpr int BK = 128 / (int)sizeof(T);
    const int E = p.E > 0 ? p.E : 1;
    const int64_t avg = max_rows / E;
    // (the band tiles address their operands with 32-bit lane offsets; slices of small weights, which come from the last-level cache,
    // keep the register-staged tiles)
    const bool band_ok = kBf16 && !p.k_count && p.K % 64 == 0 && p.a_extent_bytes != 0 && p.b_extent_bytes != 0;
    const int band_tiles = (p.N_out + (SWIGLU ? kBandCols / 2 : kBandCols) - 1) / (SWIGLU ? kBandCols / 2 : kBandCols);
    if constexpr (kBf16 && !SWIGLU && std::is_same<TO, float>::value) {
        if (p.k_splits > 1 && band_ok && p.k_slice % 64 == 0 &&
            (E == 1 ? max_rows > 32 : ((int64_t)E * p.N_out * p.K >= 1 << 24 && avg > 20 && band_groups(E, max_rows, band_tiles, p.k_splits, false) &&
                                      !SliceEstimate(E, max_rows, p.N_out, p.K).large_beats_band(p.k_splits))))
            return {Route::kBandSlices};
    }
    if constexpr (!SWIGLU) {
        // K in slices over workgroups: 32-row tiles, 64-row tiles where up to 64 rows can stream the weights once
        if (p.k_splits > 1) {
            if constexpr (kBf16) {
                if (E > 1 && avg > 20 && p.k_slice % 64 == 0 && p.a_extent_bytes != 0 && p.b_extent_bytes != 0 && !p.k_count &&
                    large_slice_tile(E, max_rows, p.N_out, p.k_slice * p.k_splits, p.k_splits))
                    return {Route::kSlices256};
            }
            return {avg > 32 ? Route::kSlices64 : Route::kSlices32};
        }
    }
    // (Float32 results of up to 192 rows keep the kernels that add K up in four chains: 16 x [2048, 5632], 48 rows, 2.2e-7 off, in the band
    // tiles' one chain 4.7e-7, as the 256-row tile's; in bfloat16 results, 1.7e-3 off, neither shows.)
    if constexpr (kBf16) {
        if (band_ok && (avg > 192 || !std::is_same<TO, float>::value)) {
            if (E > 1 && band_groups(E, max_rows, band_tiles, 1, SWIGLU)) return {Route::kBand};
            if constexpr (!SWIGLU) {
                if (E == 1 && band_dense(max_rows, p.N_out, p.K)) return {Route::kBand};
            }
        }
    }
    // (with a K per group, p.K is the bound on their sum)
    const int nk = p.k_count ? (p.K / E + BK - 1) / BK : (p.K + BK - 1) / BK;
    if constexpr (kBf16 && !SWIGLU && std::is_same<TO, bf16_t>::value) {
        // weight gradients over up to 512 padded rows per group that are large enough to fill the chip four deep
        if (p.k_count && !p.a_rows && nk <= 8 && (int64_t)E * ((avg + kShortBM - 1) / kShortBM) * ((p.N_out + kShortBN - 1) / kShortBN) >= 2048)
            return {Route::kShort};
    }
    // Few rows per group: a stream of weights (E == 1: the row count is exact; several groups vary around their mean, and
    // a group beyond 32 rows reads its weights twice).  Measured, microseconds, weights from HBM, against the register-
    // staged 32-row tiles with two slabs in flight that this kernel replaced:
    //   8 experts top-2, gate/up [28672, 4096]: 1 token 93 -> 77, 20 tokens 315 -> 271 (6.9 TB/s), 64 tokens 317 -> 289
    //   64 experts top-6, gate/up [2816, 2048]: 3 tokens 51 -> 39, 20 tokens 134 -> 104, 64 tokens 144 -> 117
    //   down [4096, 14336]: 1 token 142 -> 43, 20 tokens 178 -> 141, 64 tokens 179 -> 157
    //   128 tokens (32 rows per expert), gate/up: 430 against 343 with 256-row tiles, hence the bound.
    const int pieces = (int)(((int64_t)p.K * (int)sizeof(T) + 255) / 256);
    if (avg <= (E == 1 ? 32 : 20) && p.N_out >= 32 && !p.k_count) {
        // (tiles of 16 activation rows for few rows per group: half of the registers for them; gate/up [2816, 2048] x 64, 24 tokens
        // with the down projection 179 -> 175 us, [28672, 4096] x 8, 1 token 129.5 -> 126.5.  A group beyond 16 rows reads its weights
        // twice: 8 experts with 16 rows each 457 -> 555 us, hence the bound well below them.)
        const int mt = avg <= 4 ? 1 : 2;
        if constexpr (SWIGLU) return {Route::kStream, 2, mt, 4};
        else {
            // Eight waves split K where there are at least four pieces for each (a panel of 16 rows then reads 2 KB of
            // every row per step): [4096, 4096] x 16 rows 10.3 us against 11.7 with four waves and 14.5 with four waves
            // and 32 rows.  With more rows per group the activations, read once per panel, ask for panels of 32 rows
            // (8 experts x 16 rows, [4096, 14336]: 157 against 167).  A short K keeps four waves (64 experts, [2048, 1408],
            // 3 tokens: 23 against 37 us).
            const int64_t groups = max_rows < E ? max_rows : E;
            if (pieces >= 32 && (pieces >= 64 || groups * p.N_out <= 16 * 1024)) return {Route::kStream, E == 1 || avg <= 8 ? 1 : 2, mt, 8};
            return {Route::kStream, groups * p.N_out < 32 * 256 ? 1 : 2, mt, 4};
        }
    }
    if constexpr (!SWIGLU) {
        if (streams_long_k(avg, pieces, p.N_out) && !p.k_count) return {Route::kStream, 2, 4, 4};
    }
    switch (pick_group_tile<kBf16, SWIGLU>(max_rows, E, p.N_out, nk)) {
        case GroupTile::kSmall32: return {Route::kSmall32};
        case GroupTile::kSmall64: return {Route::kSmall64};
        case GroupTile::kSeq: return {Route::kSeq};
        case GroupTile::kMid: return {Route::kMid};
        default: return {Route::kBig};
    }
}

template <typename T, typename TO, bool SWIGLU>
static int launch_grouped(const GroupedArgs& p, int64_t max_rows, hipStream_t s) {
    constexpr bool kBf16 = std::is_same<T, bf16_t>::value, kF32Out = std::is_same<TO, float>::value;
    const GroupedRoute r = grouped_route<T, TO, SWIGLU>(p, max_rows);
    switch (r.kernel) {
        case Route::kBandSlices:
            if constexpr (kBf16 && !SWIGLU && kF32Out)
                return launch_band<TO, false, true>(p, max_rows, p.E <= 1 ? band_height(max_rows, p.N_out, p.K, p.k_splits) : kBandRows, s);
            break;
        case Route::kSlices256:
            if constexpr (kBf16 && !SWIGLU) return launch_mid_sliced<>(p, max_rows, s);
            break;
        case Route::kSlices64:
            if constexpr (!SWIGLU) return launch_cfg<T, TO, 64, 128, 1, 4, 1, 32, SWIGLU>(p, max_rows, s);
            break;
        case Route::kSlices32:
            if constexpr (!SWIGLU) return launch_cfg<T, TO, 32, 128, 1, 4, 1, 32, SWIGLU>(p, max_rows, s);
            break;
        case Route::kBand:
            if constexpr (kBf16) return launch_band<TO, SWIGLU, false>(p, max_rows, p.E <= 1 ? band_height(max_rows, p.N_out, p.K, 1) : kBandRows, s);
            break;
        case Route::kShort:
            if constexpr (kBf16 && !SWIGLU && !kF32Out) return launch_short(p, max_rows, s);
            break;
        case Route::kStream: {
            auto panels = [&](auto np, auto kw) {
                constexpr int NP = decltype(np)::value, KW = decltype(kw)::value;
                return r.mt == 1 ? launch_stream<T, TO, NP, 1, KW, SWIGLU>(p, max_rows, s) : launch_stream<T, TO, NP, 2, KW, SWIGLU>(p, max_rows, s);
            };
            typedef std::integral_constant<int, 1> One;
            typedef std::integral_constant<int, 2> Two;
            typedef std::integral_constant<int, 4> Four;
            typedef std::integral_constant<int, 8> Eight;
            if constexpr (SWIGLU) return panels(Two{}, Four{});
            else {
                if (r.mt == 4) return launch_stream<T, TO, 2, 4, 4, SWIGLU>(p, max_rows, s);
                if (r.kw == 8) return r.np == 1 ? panels(One{}, Eight{}) : panels(Two{}, Eight{});
                return r.np == 1 ? panels(One{}, Four{}) : panels(Two{}, Four{});
            }
        }
        case Route::kSmall32: return launch_small<T, TO, 1, SWIGLU ? 2 : 1, 4, 1, SWIGLU>(p, max_rows, s);
        case Route::kSmall64: return launch_small<T, TO, 2, 2, 4, 1, SWIGLU>(p, max_rows, s);
        case Route::kSeq:
            if constexpr (!kBf16) return launch_small<T, TO, 1, SWIGLU ? 2 : 1, 1, 2, SWIGLU>(p, max_rows, s);
            break;
        case Route::kMid:
            if constexpr (SWIGLU) return launch_cfg<T, TO, 128, 128, 2, 2, 4, 8, SWIGLU>(p, max_rows, s);
            else return launch_cfg<T, TO, 128, 256, 2, 4, 4, 8, SWIGLU>(p, max_rows, s);
        case Route::kBig: break;
    }
    // 256 x 256 tile, 8 waves (2 per SIMD: one wave's LDS / memory waits are covered by the other's MFMAs), 128
    // accumulator registers per lane.
    return launch_cfg<T, TO, 256, 256, 2, 4, 4, 8, SWIGLU, true>(p, max_rows, s);
}

static bool extent32_ok(int64_t rows, int64_t row_elems, int elem_size) {
    return rows > 0 && rows <= (int64_t)0xffffffffLL / (row_elems * elem_size);
}

// Training forward: the prefill tile of the direct-to-LDS kernel with both outputs.  Other group sizes and
// operands beyond 32-bit lane offsets take the two-kernel route (plain product, then silu(g) * u).
constexpr int64_t kSaveGuMinAvgRows = 768;
template <typename T>
static bool gateup_save_supported(int64_t a_rows_total, int E, int64_t max_rows, int H, int I) {
    constexpr int BK = 128 / (int)sizeof(T);
    if (E <= 0 || max_rows / E <= kSaveGuMinAvgRows || H % BK != 0 || I % (16 / (int)sizeof(T)) != 0) return false;
    return extent32_ok(a_rows_total, H, (int)sizeof(T)) && extent32_ok(2 * (int64_t)I, H, (int)sizeof(T));
}

template <typename T>
static int launch_gateup_save(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    constexpr int BM = 256, BN = 256;
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + BN / 2 - 1) / (BN / 2);
    constexpr size_t smem = dma_lds_bytes(BM, BN);
    auto kern = [] {
        if constexpr (std::is_same<T, bf16_t>::value) return grouped_gemm_dma16_kernel<T, 4, 8, true, true>;
        else return grouped_gemm_dma_kernel<T, T, BM, BN, 2, 4, 4, 8, true, true>;
    }();
    static LdsReservation reserved;
    hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern)}, (int)smem);
    if (e != hipSuccess) {
        set_error("grouped GEMM: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
        return ATS_ERR_LAUNCH;
    }
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = max_rows / (p.E > 0 ? p.E : 1) >= kAlignedBandsMinAvgRows ? 1 : 0;
    const int64_t blocks = grid_blocks(max_rows, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(512), smem, s, p);
    return ATS_OK;
}

// Training backward: dh = dy . Wd with the SwiGLU gradient in the epilogue (prefill tile of the direct-to-LDS kernel).
constexpr int64_t kDsiluMinAvgRows = 256;
template <typename T>
static bool down_dgrad_dsilu_supported(int E, int64_t max_rows, int H, int I) {
    constexpr int BK = 128 / (int)sizeof(T);
    if (E <= 0 || max_rows / E <= kDsiluMinAvgRows || H % BK != 0 || I % (16 / (int)sizeof(T)) != 0) return false;
    return extent32_ok(I, H, (int)sizeof(T));
}

template <typename T>
static int launch_down_dgrad_dsilu(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    constexpr int BM = 256, BN = 256;
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + BN - 1) / BN;
    constexpr size_t smem = dma_lds_bytes(BM, BN);
    auto kern = [] {
        if constexpr (std::is_same<T, bf16_t>::value) return grouped_gemm_dma16_kernel<T, 4, 8, false, false, true>;
        else return grouped_gemm_dma_kernel<T, T, BM, BN, 2, 4, 4, 8, false, false, true>;
    }();
    static LdsReservation reserved;
    hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern)}, (int)smem);
    if (e != hipSuccess) {
        set_error("grouped GEMM: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
        return ATS_ERR_LAUNCH;
    }
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = max_rows / (p.E > 0 ? p.E : 1) >= kAlignedBandsMinAvgRows ? 1 : 0;
    const int64_t blocks = grid_blocks(max_rows, p.E, BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(512), smem, s, p);
    return ATS_OK;
}

// Products against weights stored [K][N] (the forward's own weights in the backward's data gradients): the
// prefill tile of the bfloat16 direct-to-LDS kernel only; other group sizes and types multiply by a transposed copy.
static bool kmajor_supported(int E, int64_t max_rows, int N, int K, int64_t ldb, int64_t min_avg_rows) {
    if (E <= 0 || max_rows / E <= min_avg_rows || K % 64 != 0 || N % 8 != 0 || N < 8 || ldb % 8 != 0 || ldb < N) return false;
    return extent32_ok(K, ldb, 2);
}

template <typename TO, bool DSILU>
static int launch_kmajor(const GroupedArgs& p0, int64_t max_rows, hipStream_t s) {
    constexpr int BM = 256, BN = 256;
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + BN - 1) / BN;
    constexpr size_t smem = dma_lds_bytes(BM, BN);
    auto kern = grouped_gemm_dma16_kernel<TO, 4, 8, false, false, DSILU, true>;
    auto kern_mid = grouped_gemm_dma16_kernel<TO, 4, 8, false, false, DSILU, true, !DSILU>;
    static LdsReservation reserved;
    hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern), reinterpret_cast<const void*>(kern_mid)}, (int)smem);
    if (e != hipSuccess) {
        set_error("grouped GEMM: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
        return ATS_ERR_LAUNCH;
    }
    p.sm = 4;
    p.sn = 8;
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = max_rows / (p.E > 0 ? p.E : 1) >= kAlignedBandsMinAvgRows ? 1 : 0;
    if (!DSILU && p.E == 1) p.tile_rows = dense_tile_rows(max_rows, p.n_tiles, p.K / 64, p.sm, p.sn);
    const int64_t blocks = grid_blocks(max_rows, p.E, p.tile_rows ? p.tile_rows : BM, p.n_tiles, p.sm, p.sn, p.aligned_bands != 0);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(p.tile_rows || mid_rows(max_rows, p.E) ? kern_mid : kern, dim3((unsigned)blocks), dim3(512), smem, s, p);
    return ATS_OK;
}

// Supertiles that the busiest XCD takes, one after another: the time of a tile for each, however few tiles they hold, since tiles
// at the same place of a supertile run on the same CU (32 rows x 4096 columns are 16 supertiles of 8 x 4 tiles with one row of
// tiles each: twice the time of 2048 columns).
static int64_t xcd_rounds(int64_t m_tiles, int n_tiles) {
    int sm, sn;
    pick_supertile(n_tiles, &sm, &sn);
    return ((m_tiles + sm - 1) / sm * ((n_tiles + sn - 1) / sn) + kNumXcd - 1) / kNumXcd;
}
static float rounds_time(const TileCost& c, int64_t max_rows, int E, int n_cols, int k_slabs) {
    const int64_t avg = (max_rows + E - 1) / E;
    return xcd_rounds(E * ((avg + c.rows - 1) / c.rows), (n_cols + c.cols - 1) / c.cols) * (k_slabs * c.per_slab + c.per_tile);
}

// Float32 products against K-major operands on the small tiles, in microseconds, and what a transposing pass costs.  The
// tiles' constants are those of launch_grouped, a tenth more per slab for the 4-byte fragment reads (and less per tile for
// short sums, of which several share a CU).  Copies and their product -> operands as they lie:
//   weight gradients, rows x [M, N]: 512 x [512, 512] 47 -> 8; 2000 x [512, 512] 75 -> 21; 2048 x [2048, 2048] 225 -> 162;
//     2048 x [4096, 4096] 503 (650); 8 x 128 x [2816, 512] 63 -> 46; 8 x 500 x [2816, 512] 153 -> 132; 8 x 500 x [4096, 1024] 299 (355)
//   data gradients, rows x [N, K]: 512 x [512, 1024] 41 -> 11; 2000 x [512, 1024] 41 -> 29; 2048 x [2048, 2048] 209 -> 160;
//     4096 x [4096, 4096] 961 (1196); 8 x 128 x [512, 2816] 56 -> 37; 8 x 250 x [1408, 512] 61 -> 43
static float small_kmajor_time(int64_t max_rows, int E, int N, int K) {
    const int nk = (K + 31) / 32;
    const float t32 = tile_time(TileCost{32, 32, 0.20f, 1.5f, 1}, max_rows, E, N, nk);
    const float t64 = tile_time(TileCost{64, 64, 0.64f, 1.6f, 1}, max_rows, E, N, nk);
    return t64 < t32 ? t64 : t32;
}
// The product of copies: their passes at 4 TB/s and 4 us each, then the least of the tiles that launch_grouped has for it.
static float transposed_time(int64_t max_rows, int E, int N, int K, int64_t copied, int copies) {
    const int nk = (K + 31) / 32;
    float best = tile_time(TileCost{256, 256, 7.3f, 25.f, 1}, max_rows, E, N, nk);      // (62 us for five slabs)
    for (const TileCost& c : {TileCost{128, 256, 3.65f, 5.f, 1}, TileCost{64, 64, 0.58f, 3.f, 1}, TileCost{32, 32, 0.18f, 1.5f, 1}}) {
        const float t = tile_time(c, max_rows, E, N, nk);
        if (t < best) best = t;
    }
    return best + (float)copied * 8.f / 4e6f + 4.f * copies;
}
// 64 rows and columns per tile, or 32 (the same bits)?  Groups of unequal rows (uneven) end in half a tile on average, which
// decides where a CU gets two or three tiles; a CU holds four workgroups of the small tile, two of the large one.  The constants
// reproduce these within a tenth, microseconds with 64 | 32:
//   weight gradients, 8 groups, rows in all x [2816, 512]: 500 51 | 43, 1024 64 | 59, 2000 98 | 91, 4000 145 | 153 (second operand
//     gathered; with the row numbers read where they are needed instead of a slab ahead 56, 72, 117, 192 in 64 rows)
//   data gradients, 8 groups, rows in all x [512, 2816]: 1024 51 | 51, 2000 113 | 80, 4000 170 | 142; x [1408, 512]: 1024 39 | 26,
//     2000 50 | 43, 4000 81 | 76; one group 2048 x [2048, 2048] 166 | 175
static bool kmajor_wide(int64_t max_rows, int E, int N, int K, bool uneven) {
    const int nk = (K + 31) / 32;
    const double avg = (double)max_rows / E;
    auto time = [&](int tile, double per_slab, double per_tile, int min_tiles) {
        const double rows = uneven ? avg / tile + 0.5 : (double)(((int64_t)ceil(avg) + tile - 1) / tile);
        const int64_t per_cu = (int64_t)ceil(E * rows * ((N + tile - 1) / tile) / 256.);
        return (per_cu > min_tiles ? per_cu : min_tiles) * (nk * per_slab + per_tile);
    };
    return time(64, 0.62, 3.3, 1) < time(32, 0.17, 0.65, 2);
}

// Weight gradient of a linear layer, out[m, n] = sum_t a[t, m] b[t, n]: tiles and slices as launch_cfg takes them for the
// product of transposed copies.
template <typename TO, bool SLICED>
static int launch_tn(const GroupedArgs& p0, int64_t rows, hipStream_t s) {
    GroupedArgs p = p0;
    p.n_tiles = (p.N_out + 255) / 256;
    constexpr size_t smem = dma_lds_bytes(256, 256);
    auto kern = grouped_gemm_dma16_kernel<TO, 4, 8, false, false, false, true, true, SLICED, true>;
    static LdsReservation reserved;
    hipError_t e = reserve_lds(reserved, {reinterpret_cast<const void*>(kern)}, (int)smem);
    if (e != hipSuccess) {
        set_error("grouped GEMM: cannot reserve %zu bytes of LDS: %s", smem, hipGetErrorString(e));
        return ATS_ERR_LAUNCH;
    }
    pick_supertile(p.n_tiles, &p.sm, &p.sn);
    p.aligned_bands = 0;
    p.tile_rows = SLICED ? 0 : dense_tile_rows(rows, p.n_tiles, (p.K + 63) / 64, p.sm, p.sn);
    const int64_t blocks = grid_blocks(rows * p.k_splits, p.k_splits, p.tile_rows ? p.tile_rows : 256, p.n_tiles, p.sm, p.sn, false);
    if (blocks > 0x7fffffffLL) {
        set_error("grouped GEMM: grid of %lld blocks", (long long)blocks);
        return ATS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(512), smem, s, p);
    return ATS_OK;
}

// Bytes reachable from a buffer descriptor, or 0 when they do not fit its 32-bit range.
static uint32_t extent32(int64_t rows, int64_t row_elems, int elem_size) {
    if (rows <= 0 || rows > (int64_t)0xffffffffLL / (row_elems * elem_size)) return 0;
    return (uint32_t)(rows * row_elems * elem_size);
}

static int check_common(const char* name, const void* a, const void* const* w, const void* out,
                        const int32_t* row_start, const int32_t* row_count, int E, int64_t max_rows, int H, int I,
                        int dtype) {
    ATS_REQUIRE(E > 0 && E <= 4096 && max_rows >= 0 && H > 0 && I > 0, ATS_ERR_INVALID_ARG,
                "%s: E=%d max_rows=%lld H=%d I=%d", name, E, (long long)max_rows, H, I);
    ATS_REQUIRE(dtype == ATS_F32 || dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "%s: dtype tag %d", name, dtype);
    ATS_REQUIRE(a && w && out && row_start && row_count, ATS_ERR_INVALID_ARG, "%s: null pointer", name);
    const int vec = dtype == ATS_F32 ? 4 : 8;
    ATS_REQUIRE(H % vec == 0 && I % vec == 0, ATS_ERR_UNSUPPORTED,
                "%s: H=%d and I=%d must be multiples of %d (16-byte rows)", name, H, I, vec);
    ATS_REQUIRE(aligned16(a) && aligned16(out), ATS_ERR_INVALID_ARG, "%s: operands must be 16-byte aligned", name);
    return ATS_OK;
}

}  // namespace ats

extern "C" int ats_grouped_gemm_route(int E, int64_t max_rows, int N, int K, int k_splits, int swiglu, int out_dtype) {
    using namespace ats;
    if (E <= 0 || max_rows <= 0 || N <= 0 || K <= 0 || k_splits < 1 || K % k_splits != 0 || (swiglu && k_splits > 1)) return -1;
    GroupedArgs p{};
    p.E = E;
    p.N_out = N;
    p.K = K;
    p.k_splits = k_splits;
    p.k_slice = K / k_splits;
    p.a_extent_bytes = p.b_extent_bytes = 0xffffffffu;
    const Route r = (swiglu ? grouped_route<bf16_t, bf16_t, true>(p, max_rows) : out_dtype == ATS_F32 ? grouped_route<bf16_t, float, false>(p, max_rows)
                                                                                                 : grouped_route<bf16_t, bf16_t, false>(p, max_rows)).kernel;
    switch (r) {
        case Route::kBand:
        case Route::kBandSlices: return ATS_ROUTE_BAND;
        case Route::kStream: return ATS_ROUTE_STREAM;
        case Route::kBig: return swiglu && K % 64 == 0 && once_weights(max_rows, E) ? ATS_ROUTE_256_ONCE : ATS_ROUTE_256;
        case Route::kSlices256: return once_slices(max_rows, E, N, K) ? ATS_ROUTE_256_ONCE : ATS_ROUTE_256;
        case Route::kMid: return ATS_ROUTE_128;
        default: return ATS_ROUTE_SMALL;
    }
}

extern "C" int ats_grouped_gateup_swiglu_save_supported(int64_t a_num_rows, int E, int64_t max_rows, int H, int I,
                                                        int dtype) {
    using namespace ats;
    if (H <= 0 || I <= 0) return 0;
    if (dtype == ATS_F32) return gateup_save_supported<float>(a_num_rows, E, max_rows, H, I) ? 1 : 0;
    if (dtype == ATS_BF16) return gateup_save_supported<bf16_t>(a_num_rows, E, max_rows, H, I) ? 1 : 0;
    return 0;
}

// The optional transposed copy of a training launch: bf16 only, a 16-byte aligned buffer whose row stride holds
// every group's padded columns (ats_wgrad_padded_rows), and the groups' first columns from ats_wgrad_plan.
static int check_transposed(const char* name, const void* t_out, int64_t ld_t, const int32_t* t_col0, int64_t max_rows,
                            int E, int dtype) {
    if (!t_out) return ATS_OK;
    ATS_REQUIRE(dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "%s: the transposed copy is written for bfloat16 only", name);
    ATS_REQUIRE(t_col0 && ats::aligned16(t_out) && ld_t % 64 == 0 && ld_t >= ats_wgrad_padded_rows(max_rows, E),
                ATS_ERR_INVALID_ARG, "%s: transposed copy needs the groups' first columns, a 16-byte aligned buffer and "
                "a row stride that is a multiple of 64 and at least %lld (got %lld)", name,
                (long long)ats_wgrad_padded_rows(max_rows, E), (long long)ld_t);
    return ATS_OK;
}

extern "C" int ats_grouped_gateup_swiglu_save(const void* a, int64_t a_num_rows, const int32_t* a_rows, int a_row_div,
                                              const void* const* w_gu, void* h, void* gu, const int32_t* row_start,
                                              const int32_t* row_count, int E, int64_t max_rows, int H, int I,
                                              int dtype, void* h_t, int64_t ld_t, const int32_t* t_col0,
                                              ats_stream_t stream) {
    using namespace ats;
    int rc = check_common("ats_grouped_gateup_swiglu_save", a, w_gu, h, row_start, row_count, E, max_rows, H, I, dtype);
    if (rc != ATS_OK) return rc;
    rc = check_transposed("ats_grouped_gateup_swiglu_save", h_t, ld_t, t_col0, max_rows, E, dtype);
    if (rc != ATS_OK) return rc;
    ATS_REQUIRE(gu && aligned16(gu), ATS_ERR_INVALID_ARG, "ats_grouped_gateup_swiglu_save: gu must be a 16-byte aligned buffer");
    ATS_REQUIRE(a_num_rows > 0 && (!a_rows || a_row_div > 0), ATS_ERR_INVALID_ARG,
                "ats_grouped_gateup_swiglu_save: a_row_div=%d a_num_rows=%lld", a_row_div, (long long)a_num_rows);
    ATS_REQUIRE(ats_grouped_gateup_swiglu_save_supported(a_num_rows, E, max_rows, H, I, dtype), ATS_ERR_UNSUPPORTED,
                "ats_grouped_gateup_swiglu_save: needs more than %lld rows per expert on average, H a multiple of the "
                "K slab and operands within 4 GiB (E=%d max_rows=%lld H=%d I=%d); use the plain product and "
                "ats_silu_mul_fwd", (long long)kSaveGuMinAvgRows, E, (long long)max_rows, H, I);
    GroupedArgs p{};
    p.a = a;
    p.a_rows = a_rows;
    p.a_row_div = a_rows ? a_row_div : 1;
    p.lda = H;
    p.b = w_gu;
    p.ldb = H;
    p.out = h;
    p.ldo = I;
    p.gu_out = gu;
    p.ld_gu = 2 * (int64_t)I;
    p.t_out = h_t;
    p.ld_t = ld_t;
    p.t_col0 = t_col0;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = H;
    p.N_out = I;
    p.up_offset = I;
    const int es = dtype == ATS_F32 ? 4 : 2;
    p.a_extent_bytes = extent32(a_num_rows, H, es);
    p.b_extent_bytes = extent32(2 * (int64_t)I, H, es);
    hipStream_t s = as_stream(stream);
    rc = dtype == ATS_F32 ? launch_gateup_save<float>(p, max_rows, s) : launch_gateup_save<bf16_t>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH("ats_grouped_gateup_swiglu_save");
    return ATS_OK;
}

extern "C" int ats_grouped_down_dgrad_dsilu_supported(int E, int64_t max_rows, int H, int I, int dtype) {
    using namespace ats;
    if (H <= 0 || I <= 0) return 0;
    if (dtype == ATS_F32) return down_dgrad_dsilu_supported<float>(E, max_rows, H, I) ? 1 : 0;
    if (dtype == ATS_BF16) return down_dgrad_dsilu_supported<bf16_t>(E, max_rows, H, I) ? 1 : 0;
    return 0;
}

extern "C" int ats_grouped_down_dgrad_dsilu(const void* dy, const void* const* w_dT, const void* gu, void* dgu,
                                            const int32_t* row_start, const int32_t* row_count, int E,
                                            int64_t max_rows, int H, int I, int dtype, void* dgu_t, int64_t ld_t,
                                            const int32_t* t_col0, ats_stream_t stream) {
    using namespace ats;
    int rc = check_common("ats_grouped_down_dgrad_dsilu", dy, w_dT, dgu, row_start, row_count, E, max_rows, H, I, dtype);
    if (rc != ATS_OK) return rc;
    rc = check_transposed("ats_grouped_down_dgrad_dsilu", dgu_t, ld_t, t_col0, max_rows, E, dtype);
    if (rc != ATS_OK) return rc;
    ATS_REQUIRE(gu && aligned16(gu), ATS_ERR_INVALID_ARG, "ats_grouped_down_dgrad_dsilu: gu must be a 16-byte aligned buffer");
    ATS_REQUIRE(ats_grouped_down_dgrad_dsilu_supported(E, max_rows, H, I, dtype), ATS_ERR_UNSUPPORTED,
                "ats_grouped_down_dgrad_dsilu: needs more than %lld rows per expert on average, H a multiple of the K "
                "slab and one expert's weights within 4 GiB (E=%d max_rows=%lld H=%d I=%d); use ats_grouped_gemm_nt and "
                "ats_silu_mul_bwd", (long long)kDsiluMinAvgRows, E, (long long)max_rows, H, I);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = dy;
    p.a_row_div = 1;
    p.lda = H;
    p.b = w_dT;
    p.ldb = H;
    p.out = dgu;
    p.ldo = 2 * (int64_t)I;
    p.gu_out = const_cast<void*>(gu);
    p.ld_gu = 2 * (int64_t)I;
    p.t_out = dgu_t;
    p.ld_t = ld_t;
    p.t_col0 = t_col0;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = H;
    p.N_out = I;
    p.up_offset = I;
    const int es = dtype == ATS_F32 ? 4 : 2;
    p.a_extent_bytes = 0xffffffffu;       // the descriptor starts at the tile's first row
    p.b_extent_bytes = extent32(I, H, es);
    hipStream_t s = as_stream(stream);
    rc = dtype == ATS_F32 ? launch_down_dgrad_dsilu<float>(p, max_rows, s) : launch_down_dgrad_dsilu<bf16_t>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH("ats_grouped_down_dgrad_dsilu");
    return ATS_OK;
}

extern "C" int ats_grouped_down_dgrad_dsilu_nn_supported(int E, int64_t max_rows, int H, int I, int dtype) {
    using namespace ats;
    if (H <= 0 || I <= 0 || dtype != ATS_BF16) return 0;
    return kmajor_supported(E, max_rows, I, H, I, kDsiluMinAvgRows) ? 1 : 0;
}
extern "C" int ats_grouped_down_dgrad_dsilu_nn(const void* dy, const void* const* w_d, const void* gu, void* dgu,
                                               const int32_t* row_start, const int32_t* row_count, int E,
                                               int64_t max_rows, int H, int I, int dtype, void* dgu_t, int64_t ld_t,
                                               const int32_t* t_col0, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_down_dgrad_dsilu_nn";
    int rc = check_common(name, dy, w_d, dgu, row_start, row_count, E, max_rows, H, I, dtype);
    if (rc != ATS_OK) return rc;
    rc = check_transposed(name, dgu_t, ld_t, t_col0, max_rows, E, dtype);
    if (rc != ATS_OK) return rc;
    ATS_REQUIRE(gu && aligned16(gu), ATS_ERR_INVALID_ARG, "%s: gu must be a 16-byte aligned buffer", name);
    ATS_REQUIRE(ats_grouped_down_dgrad_dsilu_nn_supported(E, max_rows, H, I, dtype), ATS_ERR_UNSUPPORTED,
                "%s: bfloat16 with more than %lld rows per expert on average, H a multiple of 64, I of 8 and one expert's "
                "weights within 4 GiB (E=%d max_rows=%lld H=%d I=%d dtype=%d); use ats_grouped_down_dgrad_dsilu on "
                "transposed weights", name, (long long)kDsiluMinAvgRows, E, (long long)max_rows, H, I, dtype);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = dy;
    p.a_row_div = 1;
    p.lda = H;
    p.b = w_d;
    p.ldb = I;
    p.out = dgu;
    p.ldo = 2 * (int64_t)I;
    p.gu_out = const_cast<void*>(gu);
    p.ld_gu = 2 * (int64_t)I;
    p.t_out = dgu_t;
    p.ld_t = ld_t;
    p.t_col0 = t_col0;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = H;
    p.N_out = I;
    p.up_offset = I;
    p.a_extent_bytes = 0xffffffffu;       // the descriptor starts at the tile's first row
    p.b_extent_bytes = extent32(H, I, 2);
    rc = launch_kmajor<bf16_t, true>(p, max_rows, as_stream(stream));
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_grouped_gemm_nn_supported(int E, int64_t max_rows, int N, int K, int64_t ldb, int dtype) {
    using namespace ats;
    if (N <= 0 || K <= 0 || dtype != ATS_BF16) return 0;
    return kmajor_supported(E, max_rows, N, K, ldb, 192) ? 1 : 0;
}
extern "C" int ats_grouped_gemm_nn(const void* a, int64_t lda, int64_t a_num_rows, const int32_t* a_rows, int a_row_div,
                                   const void* const* b_ptrs, int64_t ldb, void* out, int64_t ldo,
                                   const int32_t* row_start, const int32_t* row_count, int E, int64_t max_rows, int N,
                                   int K, int dtype, int out_dtype, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_gemm_nn";
    ATS_REQUIRE(E > 0 && E <= 4096 && max_rows >= 0 && N > 0 && K > 0, ATS_ERR_INVALID_ARG,
                "%s: E=%d max_rows=%lld N=%d K=%d", name, E, (long long)max_rows, N, K);
    ATS_REQUIRE(dtype == ATS_BF16 && (out_dtype == ATS_F32 || out_dtype == ATS_BF16), ATS_ERR_UNSUPPORTED,
                "%s: dtype tags %d -> %d (bfloat16 operands, bfloat16 or float32 out)", name, dtype, out_dtype);
    ATS_REQUIRE(a && b_ptrs && out && row_start && row_count, ATS_ERR_INVALID_ARG, "%s: null pointer", name);
    ATS_REQUIRE(!a_rows || (a_row_div > 0 && a_num_rows > 0), ATS_ERR_INVALID_ARG, "%s: a_row_div=%d a_num_rows=%lld",
                name, a_row_div, (long long)a_num_rows);
    const int ovec = out_dtype == ATS_F32 ? 4 : 8;
    ATS_REQUIRE(lda % 8 == 0 && lda >= K && N % ovec == 0 && ldo % ovec == 0 && ldo >= N, ATS_ERR_UNSUPPORTED,
                "%s: K=%d N=%d lda=%lld ldo=%lld must describe 16-byte aligned rows", name, K, N, (long long)lda,
                (long long)ldo);
    ATS_REQUIRE(aligned16(a) && aligned16(out), ATS_ERR_INVALID_ARG, "%s: operands must be 16-byte aligned", name);
    ATS_REQUIRE(ats_grouped_gemm_nn_supported(E, max_rows, N, K, ldb, dtype), ATS_ERR_UNSUPPORTED,
                "%s: more than 192 rows per expert on average, K a multiple of 64, N and ldb of 8 and one expert's weights "
                "within 4 GiB (E=%d max_rows=%lld N=%d K=%d ldb=%lld); use ats_grouped_gemm_nt on transposed weights", name,
                E, (long long)max_rows, N, K, (long long)ldb);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = a;
    p.a_rows = a_rows;
    p.a_row_div = a_rows ? a_row_div : 1;
    p.lda = lda;
    p.b = b_ptrs;
    p.ldb = ldb;
    p.out = out;
    p.ldo = ldo;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = K;
    p.N_out = N;
    p.up_offset = 0;
    p.a_extent_bytes = a_rows ? extent32(a_num_rows, lda, 2) : 0xffffffffu;
    p.b_extent_bytes = extent32(K, ldb, 2);
    ATS_REQUIRE(p.a_extent_bytes != 0, ATS_ERR_UNSUPPORTED, "%s: the gathered operand must stay within 4 GiB", name);
    hipStream_t s = as_stream(stream);
    const int rc = out_dtype == ATS_F32 ? launch_kmajor<float, false>(p, max_rows, s)
                                        : launch_kmajor<bf16_t, false>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

// small: the slices that fill the chip with the small tiles (1: none are needed)
extern "C" int ats_down_k_slices(int E, int64_t max_rows, int N, int K, int small) {
    using namespace ats;
    if (E <= 0 || max_rows <= 0 || N <= 0 || K <= 0 || small < 1) return 1;
    const SliceEstimate t(E, max_rows, N, K);
    auto band = [&](int s) {
        return E > 1 && max_rows / E > 20 && K % (s * 64) == 0 && band_groups(E, max_rows, (N + kBandCols - 1) / kBandCols, s, false) &&
               !t.large_beats_band(s);
    };
    float best = band(1) ? t.band(1) : t.plain();
    int slices = 1;
    if (small > 1 && !band(small) && t.small(small) <= best) {
        best = t.small(small);
        slices = small;
    }
    for (int s = 2; s <= 16 && K % (s * 64) == 0 && K / s >= 512; s *= 2) {
        const bool on_band = band(s);
        if (!on_band && !large_slice_tile(E, max_rows, N, K, s)) continue;
        // (0.7: against another fit than its own; 8 x [1024, 2048], 44 rows 16.6 us plain, 17.3 in four slices)
        const float time = on_band ? t.band(s) + (band(1) ? 0.f : 0.7f) : t.large_beats_band(s) ? 0.93f * (t.large(s) + 2.f) : t.large_with_margin(s);
        if (time < best) {
            best = time;
            slices = s;
        }
    }
    return slices;
}

// Slices of K of a bfloat16 linear layer (1: plain), by the estimated times.
extern "C" int ats_linear_k_slices(int64_t rows, int N, int K) {
    using namespace ats;
    if (rows <= 32 || rows > 256 || N <= 0 || K <= 0 || K % 64 != 0) return 1;
    // (against a long K slices on the band tiles are as fast as the small tiles: [4096, 4096] x 100 rows 19 and 20 us, 128 rows 22 and 21;
    // and a rotation behind the product adds them up on its way)
    float best = band_time(rows, N, K, 1, band_height(rows, N, K, 1));
    if (K <= 2048 || rows > 192) best = fminf(best, other_dense_time(rows, N, K));
    // (below that the second launch is what a caller waits for: [2048, 2048] x 40 rows 8.9 plain, 10.1 in slices behind other launches,
    // 10.9 and 9.8 each by itself)
    if (best < 13.f) return 1;
    int slices = 1;
    for (int s = 2; s <= 8 && K % (s * 64) == 0 && K / s >= 256; s *= 2) {
        const float t = band_time(rows, N, K, s, band_height(rows, N, K, s));
        if (t < best) {
            best = t;
            slices = s;
        }
    }
    return slices;
}

// Slices of K with which a product against [K][N] weights is to run, 0 where multiplying by a transposed copy is the
// faster one or the only one.  Above 256 rows per group it is ats_grouped_gemm_nn.  Below, the 256-column tiles of a few
// experts leave CUs idle, so K is cut (launch_mid_sliced); the estimate holds both routes against each other: a CU takes
// 1.3 us per slab and 7 per tile, partial results are written and read at 5 TB/s, a copy is made at 5.2 TB/s and
// multiplied at 4.6.  Training pass of 8 experts, top 2, [28672, 4096] and [4096, 14336], copies -> this: 256 tokens 3445 ->
// 2124 us, 588 tokens 3851 -> 2557, 760 tokens 4050 -> 2742 (the copies alone were 1100).
extern "C" int ats_grouped_gemm_nn_slices(int E, int64_t max_rows, int N, int K, int64_t ldb, int dtype) {
    using namespace ats;
    if (N <= 0 || K <= 0 || E <= 0 || max_rows <= 0 || dtype != ATS_BF16) return 0;
    if (!kmajor_supported(E, max_rows, N, K, ldb, -1)) return 0;
    const int64_t avg = (max_rows + E - 1) / E;
    if (max_rows / E > 256) return 1;
    const double weights = 2.0 * E * N * K;      // bytes
    const int64_t tiles = (int64_t)E * ((N + 255) / 256) * (E > 1 && avg > 232 ? 3 : 2) / 2;
    // (the unsliced launch of more than 192 rows never had a copy to make)
    double best = max_rows / E > 192 ? 1e30 : weights * (2 / 5.2e6 + 1 / 4.6e6) + 5.;
    int slices = 0;
    for (int s = 1; s <= 16; s *= 2) {
        if (s > 1 && (K % (s * 64) != 0 || K / s < 512)) break;
        const double t = (double)((tiles * s + 255) / 256) * (K / 64 / s * 1.3 + 7.) + (s > 1 ? 8. * max_rows * N * s / 5e6 + 4. : 0.);
        if (t < 0.97 * best) {
            best = t;
            slices = s;
        }
    }
    return slices;
}

// out: k_splits = 1: [rows, ldo = N] of out_dtype; more: float32 partial results [k_splits][part_rows][N].
extern "C" int ats_grouped_gemm_nn_sliced(const void* a, int64_t lda, const void* const* b_ptrs, int64_t ldb, void* out,
                                          int64_t part_rows, const int32_t* row_start, const int32_t* row_count, int E,
                                          int64_t max_rows, int N, int K, int k_splits, int dtype, int out_dtype,
                                          ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_gemm_nn_sliced";
    ATS_REQUIRE(E > 0 && E <= 4096 && max_rows >= 0 && N > 0 && K > 0 && part_rows >= max_rows, ATS_ERR_INVALID_ARG,
                "%s: E=%d max_rows=%lld part_rows=%lld N=%d K=%d", name, E, (long long)max_rows, (long long)part_rows, N, K);
    ATS_REQUIRE(dtype == ATS_BF16 && (out_dtype == ATS_F32 || (out_dtype == ATS_BF16 && k_splits == 1)), ATS_ERR_UNSUPPORTED,
                "%s: dtype tags %d -> %d (bfloat16 operands; slices give float32)", name, dtype, out_dtype);
    ATS_REQUIRE(a && b_ptrs && out && row_start && row_count, ATS_ERR_INVALID_ARG, "%s: null pointer", name);
    ATS_REQUIRE(lda % 8 == 0 && lda >= K, ATS_ERR_UNSUPPORTED, "%s: K=%d lda=%lld must describe 16-byte aligned rows", name, K,
                (long long)lda);
    ATS_REQUIRE(aligned16(a) && aligned16(out), ATS_ERR_INVALID_ARG, "%s: operands must be 16-byte aligned", name);
    ATS_REQUIRE(k_splits >= 1 && k_splits <= 64 && K % (k_splits * 64) == 0, ATS_ERR_UNSUPPORTED,
                "%s: K=%d is not %d slices of whole 64-element slabs", name, K, k_splits);
    if (max_rows == 0) return ATS_OK;
    ATS_REQUIRE(kmajor_supported(E, max_rows, N, K, ldb, -1) && max_rows / E <= 256, ATS_ERR_UNSUPPORTED,
                "%s: up to 256 rows per expert on average, N and ldb multiples of 8 and one expert's weights within 4 GiB "
                "(E=%d max_rows=%lld N=%d K=%d ldb=%lld)", name, E, (long long)max_rows, N, K, (long long)ldb);
    GroupedArgs p{};
    p.a = a;
    p.a_row_div = 1;
    p.lda = lda;
    p.b = b_ptrs;
    p.ldb = ldb;
    p.out = out;
    p.ldo = N;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = K;
    p.N_out = N;
    p.k_splits = k_splits;
    p.k_slice = K / k_splits;
    p.part_stride = part_rows * N;
    p.a_extent_bytes = 0xffffffffu;
    p.b_extent_bytes = extent32(K, ldb, 2);
    hipStream_t s = as_stream(stream);
    const int rc = k_splits > 1 ? launch_mid_sliced<true>(p, max_rows, s)
                   : out_dtype == ATS_F32 ? launch_kmajor<float, false>(p, max_rows, s)
                                          : launch_kmajor<bf16_t, false>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_grouped_gemm_nn_f32_supported(int E, int64_t max_rows, int N, int K) {
    using namespace ats;
    if (E <= 0 || max_rows <= 0 || N <= 0 || K <= 0 || N % 4 != 0 || K % 4 != 0) return 0;
    // The weights as they lie against their copies (4.6 TB/s, a launch and its host work: 11 us) and the product of these, for a few
    // rows the stream of weights.  3992 points, 1 .. 64 groups: half the time of the copies, 50 of them more than 4 % slower.  1 x 13 rows x [1408, 8192]: as they lie 90 us, copies 47; 5 rows x [1408, 6144] 69, 37; 8
    // rows x [2560, 8192] 92, 61; 8 rows x [2048, 2048] 16, 28.
    const int nk = (K + 31) / 32;
    const float t32 = rounds_time(TileCost{32, 32, 0.20f, 3.f, 1}, max_rows, E, N, nk);
    const float t64 = rounds_time(TileCost{64, 64, 0.64f, 2.5f, 1}, max_rows, E, N, nk);
    float copied = rounds_time(TileCost{256, 256, 7.3f, 25.f, 1}, max_rows, E, N, nk);
    for (const TileCost& c : {TileCost{128, 256, 3.65f, 5.f, 1}, TileCost{64, 64, 0.58f, 3.f, 1}, TileCost{32, 32, 0.18f, 1.5f, 1}})
        copied = fminf(copied, rounds_time(c, max_rows, E, N, nk));
    const float weights = (float)E * N * K * 4e-6f;
    if (max_rows / E <= (E == 1 ? 32 : 20)) copied = fminf(copied, 3.f + fmaxf(K * 0.0024f, weights / 4.5f));
    return 0.95f * fminf(t32, t64) <= copied + weights * 2.f / 4.6f + 11.f ? 1 : 0;
}
extern "C" int ats_grouped_gemm_nn_f32(const float* a, int64_t lda, const void* const* b_ptrs, int64_t ldb, float* out, int64_t ldo,
                                       const int32_t* row_start, const int32_t* row_count, int E, int64_t max_rows, int N, int K,
                                       ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_gemm_nn_f32";
    ATS_REQUIRE(E > 0 && E <= 4096 && max_rows >= 0 && N > 0 && K > 0, ATS_ERR_INVALID_ARG, "%s: E=%d max_rows=%lld N=%d K=%d",
                name, E, (long long)max_rows, N, K);
    ATS_REQUIRE(a && b_ptrs && out && row_start && row_count && aligned16(a) && aligned16(out), ATS_ERR_INVALID_ARG,
                "%s: null or misaligned pointer", name);
    ATS_REQUIRE(N % 4 == 0 && K % 4 == 0 && lda % 4 == 0 && lda >= K && ldb % 4 == 0 && ldb >= N && ldo % 4 == 0 && ldo >= N,
                ATS_ERR_UNSUPPORTED, "%s: N=%d K=%d lda=%lld ldb=%lld ldo=%lld must describe 16-byte aligned rows", name, N, K,
                (long long)lda, (long long)ldb, (long long)ldo);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = a;
    p.a_row_div = 1;
    p.lda = lda;
    p.b = b_ptrs;
    p.ldb = ldb;
    p.out = out;
    p.ldo = ldo;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = K;
    p.N_out = N;
    const int rc = kmajor_wide(max_rows, E, N, K, E > 1)
                       ? launch_small<float, float, 2, 2, 4, 1, false, false, true>(p, max_rows, as_stream(stream))
                       : launch_small<float, float, 1, 1, 4, 1, false, false, true>(p, max_rows, as_stream(stream));
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

// (max_k: bound on the sum over the groups)
extern "C" int ats_grouped_wgrad_f32_supported(int E, int64_t max_k, int M, int N) {
    using namespace ats;
    if (E <= 0 || max_k <= 0 || max_k > 0x7fffffff || M <= 0 || N <= 0 || M % 4 != 0 || N % 4 != 0) return 0;
    const int k = (int)((max_k + E - 1) / E);
    return small_kmajor_time((int64_t)E * M, E, N, k) <=
                   transposed_time((int64_t)E * M, E, N, k + 16, max_k * ((int64_t)M + N), 2) ? 1 : 0;
}
extern "C" int ats_grouped_wgrad_f32(const float* a, int64_t lda, const float* b, int64_t ldb, const int32_t* b_rows, int b_row_div,
                                     float* out, const int32_t* k_start, const int32_t* k_count, int E, int64_t max_k, int M, int N,
                                     ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_wgrad_f32";
    ATS_REQUIRE(E > 0 && E <= 4096 && max_k >= 0 && max_k <= 0x7fffffff && M > 0 && N > 0 && (E == 1 || (k_start && k_count)),
                ATS_ERR_INVALID_ARG, "%s: E=%d max_k=%lld M=%d N=%d", name, E, (long long)max_k, M, N);
    ATS_REQUIRE(a && b && out && aligned16(a) && aligned16(b) && aligned16(out) && (!b_rows || b_row_div > 0), ATS_ERR_INVALID_ARG,
                "%s: null or misaligned pointer", name);
    ATS_REQUIRE(M % 4 == 0 && N % 4 == 0 && lda % 4 == 0 && lda >= M && ldb % 4 == 0 && ldb >= N, ATS_ERR_UNSUPPORTED,
                "%s: M=%d N=%d lda=%lld ldb=%lld must describe 16-byte aligned rows", name, M, N, (long long)lda, (long long)ldb);
    GroupedArgs p{};
    p.a = a;
    p.a_row_div = 1;
    p.lda = lda;
    p.b = reinterpret_cast<const void* const*>(b);
    p.ldb = ldb;
    p.b_rows = b_rows;
    p.b_row_div = b_rows ? b_row_div : 1;
    p.out = out;
    p.ldo = N;
    p.k_start = k_start;
    p.k_count = k_count;
    p.uniform_rows = M;
    p.E = E;
    p.K = (int)max_k;
    p.N_out = N;
    const int rc = kmajor_wide((int64_t)E * M, E, N, (int)((max_k + E - 1) / E), false)
                       ? launch_small<float, float, 2, 2, 4, 1, false, true, true>(p, (int64_t)E * M, as_stream(stream))
                       : launch_small<float, float, 1, 1, 4, 1, false, true, true>(p, (int64_t)E * M, as_stream(stream));
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_wgrad_tn(const void* a, int64_t lda, const void* b, int64_t ldb, void* out, int64_t T, int M, int N,
                            int slab_slices, const int32_t* row_start, const int32_t* row_count, int dtype, int out_dtype,
                            ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_wgrad_tn";
    ATS_REQUIRE(T > 0 && T <= 0x7fffffc0 && M > 0 && N > 0 && lda >= M && ldb >= N && slab_slices >= 1 && slab_slices <= 64,
                ATS_ERR_INVALID_ARG, "%s: T=%lld M=%d N=%d lda=%lld ldb=%lld slices=%d", name, (long long)T, M, N, (long long)lda,
                (long long)ldb, slab_slices);
    ATS_REQUIRE(dtype == ATS_BF16 && (slab_slices > 1 ? out_dtype == ATS_F32 : out_dtype == ATS_BF16), ATS_ERR_UNSUPPORTED,
                "%s: dtype tags %d -> %d (bfloat16 operands; bfloat16 out, float32 with slices)", name, dtype, out_dtype);
    ATS_REQUIRE(a && b && out && row_start && row_count, ATS_ERR_INVALID_ARG, "%s: null pointer", name);
    // (offsets of a whole last slab have to fit 32 bits: a wrapped one would not be seen as lying past the end)
    const int64_t padded = (T + 63) / 64 * 64;
    ATS_REQUIRE(M % 8 == 0 && N % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && aligned16(a) && aligned16(b) && aligned16(out) &&
                    extent32_ok(padded, lda, 2) && extent32_ok(padded, ldb, 2),
                ATS_ERR_UNSUPPORTED, "%s: M=%d N=%d lda=%lld ldb=%lld must describe 16-byte aligned rows within 4 GiB", name, M,
                N, (long long)lda, (long long)ldb);
    GroupedArgs p{};
    p.a = a;
    p.a_row_div = 1;
    p.lda = lda;
    p.b = static_cast<const void* const*>(b);
    p.ldb = ldb;
    p.out = out;
    p.ldo = N;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = 1;
    p.K = (int)T;
    p.N_out = N;
    const int64_t slabs = padded / 64, per = (slabs + slab_slices - 1) / slab_slices;
    p.k_splits = (int)((slabs + per - 1) / per);
    ATS_REQUIRE(p.k_splits == slab_slices, ATS_ERR_INVALID_ARG, "%s: %lld slabs do not make %d slices", name, (long long)slabs, slab_slices);
    p.k_slice = (int)per * 64;
    p.part_stride = (int64_t)M * N;
    hipStream_t s = as_stream(stream);
    const int rc = slab_slices > 1 ? launch_tn<float, true>(p, M, s) : launch_tn<bf16_t, false>(p, M, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_grouped_gateup_swiglu(const void* a, int64_t a_num_rows, const int32_t* a_rows, int a_row_div,
                                         const void* const* w_gu, void* h, const int32_t* row_start,
                                         const int32_t* row_count, int E, int64_t max_rows, int H, int I, int dtype,
                                         ats_stream_t stream) {
    using namespace ats;
    int rc = check_common("ats_grouped_gateup_swiglu", a, w_gu, h, row_start, row_count, E, max_rows, H, I, dtype);
    if (rc != ATS_OK) return rc;
    ATS_REQUIRE(!a_rows || (a_row_div > 0 && a_num_rows > 0), ATS_ERR_INVALID_ARG,
                "ats_grouped_gateup_swiglu: a_row_div=%d a_num_rows=%lld", a_row_div, (long long)a_num_rows);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = a;
    p.a_rows = a_rows;
    p.a_row_div = a_rows ? a_row_div : 1;
    p.lda = H;
    p.b = w_gu;
    p.ldb = H;
    p.out = h;
    p.ldo = I;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = H;
    p.N_out = I;
    p.up_offset = I;
    const int es = dtype == ATS_F32 ? 4 : 2;
    p.a_extent_bytes = a_rows ? extent32(a_num_rows, H, es) : 0xffffffffu;
    p.b_extent_bytes = extent32(2 * (int64_t)I, H, es);
    hipStream_t s = as_stream(stream);
    rc = dtype == ATS_F32 ? launch_grouped<float, float, true>(p, max_rows, s)
                          : launch_grouped<bf16_t, bf16_t, true>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH("ats_grouped_gateup_swiglu");
    return ATS_OK;
}

extern "C" int ats_grouped_down(const void* h, const void* const* w_d, void* y, const int32_t* row_start,
                                const int32_t* row_count, int E, int64_t max_rows, int H, int I, int dtype,
                                int y_dtype, ats_stream_t stream) {
    using namespace ats;
    int rc = check_common("ats_grouped_down", h, w_d, y, row_start, row_count, E, max_rows, H, I, dtype);
    if (rc != ATS_OK) return rc;
    ATS_REQUIRE(y_dtype == ATS_F32 || y_dtype == dtype, ATS_ERR_UNSUPPORTED,
                "ats_grouped_down: y dtype tag %d (float32 or the operand type)", y_dtype);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = h;
    p.a_rows = nullptr;
    p.a_row_div = 1;
    p.lda = I;
    p.b = w_d;
    p.ldb = I;
    p.out = y;
    p.ldo = H;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = I;
    p.N_out = H;
    p.up_offset = 0;
    p.a_extent_bytes = 0xffffffffu;
    p.b_extent_bytes = extent32(H, I, dtype == ATS_F32 ? 4 : 2);
    hipStream_t s = as_stream(stream);
    if (dtype == ATS_F32) rc = launch_grouped<float, float, false>(p, max_rows, s);
    else if (y_dtype == ATS_F32) rc = launch_grouped<bf16_t, float, false>(p, max_rows, s);
    else rc = launch_grouped<bf16_t, bf16_t, false>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH("ats_grouped_down");
    return ATS_OK;
}

extern "C" int ats_grouped_down_splitk(const void* h, const void* const* w_d, float* parts, const int32_t* row_start,
                                       const int32_t* row_count, int E, int64_t max_rows, int64_t part_rows, int H,
                                       int I, int k_splits, int dtype, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_down_splitk";
    int rc = check_common(name, h, w_d, parts, row_start, row_count, E, max_rows, H, I, dtype);
    if (rc != ATS_OK) return rc;
    ATS_REQUIRE(k_splits >= 1 && k_splits <= 64 && part_rows >= 0, ATS_ERR_INVALID_ARG, "%s: k_splits=%d part_rows=%lld",
                name, k_splits, (long long)part_rows);
    const int slab = dtype == ATS_F32 ? 32 : 64;
    ATS_REQUIRE(I % (k_splits * slab) == 0, ATS_ERR_UNSUPPORTED, "%s: I=%d is not %d slices of whole %d-element slabs",
                name, I, k_splits, slab);
    ATS_REQUIRE(max_rows / E <= 256, ATS_ERR_UNSUPPORTED,
                "%s: %lld rows for %d experts (slices of K are built for the weight-streaming tiles, <= 256 rows per expert)",
                name, (long long)max_rows, E);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = h;
    p.a_row_div = 1;
    p.lda = I;
    p.b = w_d;
    p.ldb = I;
    p.out = parts;
    p.ldo = H;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = I;
    p.N_out = H;
    p.k_splits = k_splits;
    p.k_slice = I / k_splits;
    p.part_stride = part_rows * H;
    p.a_extent_bytes = 0xffffffffu;
    p.b_extent_bytes = extent32(H, I, dtype == ATS_F32 ? 4 : 2);
    hipStream_t s = as_stream(stream);
    rc = dtype == ATS_F32 ? launch_grouped<float, float, false>(p, max_rows, s)
                          : launch_grouped<bf16_t, float, false>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

extern "C" int ats_grouped_gemm_nt(const void* a, const void* const* a_ptrs, int64_t lda, int64_t a_num_rows,
                                   const int32_t* a_rows, int a_row_div, const void* const* b_ptrs, int64_t ldb,
                                   int64_t b_rows, void* out, int64_t ldo, const int32_t* row_start,
                                   const int32_t* row_count, const int32_t* k_count, int E, int64_t max_rows, int N,
                                   int K, int dtype, int out_dtype, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_grouped_gemm_nt";
    ATS_REQUIRE(E > 0 && E <= 4096 && max_rows >= 0 && N > 0 && K > 0, ATS_ERR_INVALID_ARG,
                "%s: E=%d max_rows=%lld N=%d K=%d", name, E, (long long)max_rows, N, K);
    ATS_REQUIRE(dtype == ATS_F32 || dtype == ATS_BF16, ATS_ERR_UNSUPPORTED, "%s: dtype tag %d", name, dtype);
    ATS_REQUIRE(out_dtype == ATS_F32 || out_dtype == dtype, ATS_ERR_UNSUPPORTED,
                "%s: out dtype tag %d (float32 or the operand type)", name, out_dtype);
    ATS_REQUIRE((a || a_ptrs) && b_ptrs && out && row_start && row_count, ATS_ERR_INVALID_ARG, "%s: null pointer", name);
    ATS_REQUIRE(!(a_ptrs && a_rows), ATS_ERR_INVALID_ARG, "%s: a gather table needs a single A base", name);
    ATS_REQUIRE(!a_rows || (a_row_div > 0 && a_num_rows > 0), ATS_ERR_INVALID_ARG, "%s: a_row_div=%d a_num_rows=%lld",
                name, a_row_div, (long long)a_num_rows);
    const int vec = dtype == ATS_F32 ? 4 : 8;
    const int ovec = out_dtype == ATS_F32 ? 4 : 8;
    ATS_REQUIRE(K % vec == 0 && lda % vec == 0 && ldb % vec == 0 && lda >= K && ldb >= K && N % ovec == 0 &&
                    ldo % ovec == 0 && ldo >= N,
                ATS_ERR_UNSUPPORTED, "%s: K=%d N=%d lda=%lld ldb=%lld ldo=%lld must describe 16-byte aligned rows", name, K, N,
                (long long)lda, (long long)ldb, (long long)ldo);
    ATS_REQUIRE((!a || aligned16(a)) && aligned16(out), ATS_ERR_INVALID_ARG, "%s: operands must be 16-byte aligned", name);
    const int slab = dtype == ATS_F32 ? 32 : 64;
    ATS_REQUIRE((!k_count && !a_ptrs) || K % slab == 0, ATS_ERR_UNSUPPORTED,
                "%s: per-expert K / A bases need K to be a multiple of %d", name, slab);
    if (max_rows == 0) return ATS_OK;
    GroupedArgs p{};
    p.a = a;
    p.a_ptrs = a_ptrs;
    p.a_rows = a_rows;
    p.a_row_div = a_rows ? a_row_div : 1;
    p.lda = lda;
    p.b = b_ptrs;
    p.ldb = ldb;
    p.k_count = k_count;
    p.out = out;
    p.ldo = ldo;
    p.row_start = row_start;
    p.row_count = row_count;
    p.E = E;
    p.K = K;
    p.N_out = N;
    p.up_offset = 0;
    const int es = dtype == ATS_F32 ? 4 : 2;
    p.a_extent_bytes = a_rows ? extent32(a_num_rows, lda, es) : 0xffffffffu;
    p.b_extent_bytes = extent32(b_rows > 0 ? b_rows : N, ldb, es);
    hipStream_t s = as_stream(stream);
    int rc;
    if (dtype == ATS_F32) rc = launch_grouped<float, float, false>(p, max_rows, s);
    else if (out_dtype == ATS_F32) rc = launch_grouped<bf16_t, float, false>(p, max_rows, s);
    else rc = launch_grouped<bf16_t, bf16_t, false>(p, max_rows, s);
    if (rc != ATS_OK) return rc;
    ATS_CHECK_LAUNCH(name);
    return ATS_OK;
}

// A linear layer: one group whose results no grouped launch has to repeat, so that float32 sums may be cut into slices of K at
// any number of rows (up to 256 launch_grouped does so itself).  Two of the 64-row workgroups share a CU: an odd third costs as
// much as a fourth.  [N, K] x rows, all of K in a wave -> slices, microseconds (half the error: four chains instead of one):
//   [1024, 512] x 512 18 -> 10, x 1000 18 -> 15, x 2000 28 -> 27; [512, 1408] x 512 40 -> 13, x 2000 40 -> 33;
//   [2048, 2048] x 257 58 -> 42, x 700 91 -> 76, x 1500 140 (147), x 2000 193 -> 160; x 4096 240 in 256-row tiles;
//   [6144, 512] x 276, three rounds of 64-row tiles on the XCDs with full bands: 41 -> 29 in 32-row ones (64-row slices 47)
extern "C" int ats_linear_nt(const void* x, const void* const* w, void* out, const int32_t* row_start, const int32_t* row_count,
                             int64_t T, int N, int K, int dtype, ats_stream_t stream) {
    using namespace ats;
    const char* name = "ats_linear_nt";
    if (dtype == ATS_F32 && T > 256 && T <= 0x7fffffff && N > 0 && K > 0 && N % 4 == 0 && K % 4 == 0 && x && w && out && row_start &&
        row_count && aligned16(x) && aligned16(out)) {
        const int nk = (K + 31) / 32;
        const int64_t rounds = xcd_rounds((T + 63) / 64, (N + 63) / 64);
        const float t64 = (float)(rounds <= 1 ? 1 : (rounds + 1) / 2 * 2) * (nk * 0.58f + 3.f);
        const float t32 = rounds_time(TileCost{32, 32, 0.18f, 1.5f, 1}, T, 1, N, nk);
        float others = rounds_time(TileCost{64, 64, 0.74f, 3.f, 1}, T, 1, N, nk);
        for (const TileCost& c : {TileCost{128, 256, 3.65f, 5.f, 1}, TileCost{256, 256, 7.3f, 7.f, 1}})
            others = fminf(others, rounds_time(c, T, 1, N, nk));
        if (t32 < others || t64 < others) {
            GroupedArgs p{};
            p.a = x;
            p.a_row_div = 1;
            p.lda = p.ldb = K;
            p.b = w;
            p.out = out;
            p.ldo = N;
            p.row_start = row_start;
            p.row_count = row_count;
            p.E = 1;
            p.K = K;
            p.N_out = N;
            const int rc = t32 <= t64 ? launch_small<float, float, 1, 1, 4, 1, false>(p, T, as_stream(stream))
                                      : launch_small<float, float, 2, 2, 4, 1, false>(p, T, as_stream(stream));
            if (rc != ATS_OK) return rc;
            ATS_CHECK_LAUNCH(name);
            return ATS_OK;
        }
    }
    return ats_grouped_gemm_nt(x, nullptr, K, T, nullptr, 1, w, K, N, out, N, row_start, row_count, nullptr, 1, T, N, K, dtype, dtype,
                               stream);
}

// Device-side view of the tile schedule: one wave per block id evaluates decode_tile_wave (the search the GEMM
// kernels run) and writes {expert, m_tile, n_tile, slice}, or -1s where the block owns no tile.
namespace ats {
__global__ __launch_bounds__(64) void debug_decode_tiles_kernel(const int32_t* __restrict__ row_count, int E, int BM,
                                                                int n_tiles, int SM, int SN, int aligned, int k_slices,
                                                                int32_t* __restrict__ out4) {
    TileCoord tc;
    int slice = 0;
    const bool ok = decode_tile_wave(blockIdx.x, row_count, E, BM, n_tiles, SM, SN, aligned != 0, &tc, k_slices, &slice);
    if (threadIdx.x == 0) {
        int32_t* o = out4 + (int64_t)blockIdx.x * 4;
        o[0] = ok ? tc.e : -1;
        o[1] = ok ? tc.mt : -1;
        o[2] = ok ? tc.nt : -1;
        o[3] = ok ? slice : -1;
    }
}
}  // namespace ats

extern "C" int ats_debug_decode_tiles_device(const int32_t* row_count_dev, int E, int BM, int n_tiles, int SM, int SN,
                                             int aligned, int k_slices, int64_t n_blocks, int32_t* out4_dev,
                                             ats_stream_t stream) {
    using namespace ats;
    ATS_REQUIRE(row_count_dev && out4_dev && E > 0 && BM > 0 && n_tiles > 0 && SM > 0 && SN > 0 && SM * SN == kSuperBlocks &&
                    k_slices >= 1 && n_blocks >= 0 && n_blocks < 0x7fffffffLL,
                ATS_ERR_INVALID_ARG, "ats_debug_decode_tiles_device: E=%d BM=%d n_tiles=%d SM=%d SN=%d k_slices=%d", E, BM,
                n_tiles, SM, SN, k_slices);
    if (n_blocks == 0) return ATS_OK;
    hipLaunchKernelGGL(debug_decode_tiles_kernel, dim3((unsigned)n_blocks), dim3(64), 0, as_stream(stream), row_count_dev,
                       E, BM, n_tiles, SM, SN, aligned, k_slices, out4_dev);
    ATS_CHECK_LAUNCH("ats_debug_decode_tiles_device");
    return ATS_OK;
}

// Host-side view of the tile schedule (for tests of the block -> tile map).
extern "C" int ats_debug_decode_tile(int64_t block, const int32_t* row_count_host, int E, int BM, int n_tiles,
                                     int SM, int SN, int aligned, int k_slices, int32_t* out4) {
    ats::TileCoord tc;
    int slice = 0;
    if (!ats::decode_tile(block, row_count_host, E, BM, n_tiles, SM, SN, aligned != 0, &tc, k_slices, &slice)) return 0;
    out4[0] = tc.e;
    out4[1] = tc.mt;
    out4[2] = tc.nt;
    out4[3] = slice;
    return 1;
}
extern "C" int64_t ats_debug_grid_blocks(int64_t max_rows, int E, int BM, int n_tiles, int SM, int SN, int aligned) {
    return ats::grid_blocks(max_rows, E, BM, n_tiles, SM, SN, aligned != 0);
}
