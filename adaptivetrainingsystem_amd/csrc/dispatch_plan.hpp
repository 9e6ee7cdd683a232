// Device parts of the dispatch plan that its kernels share: counts of a chunk, totals over chunks, ranks inside a chunk,
// and the whole plan of up to kPlanSingle assignments in one workgroup.
#pragma once
#include "ats_common.hpp"

namespace ats {

constexpr int kPlanChunk = 256;      // assignments per block of the multi-block plan (64 per wave: one step)
constexpr int kPlanSingle = 1024;    // largest plan done by one block alone (four waves: 256 each, four steps)
constexpr int kPlanMaxE = 1024;

template <typename IdxT>
__device__ __forceinline__ int load_expert(const IdxT* idx, int64_t a, int64_t n, int E, bool* bad) {
    if (a >= n) return -1;
    const long long e = (long long)idx[a];
    if (e < 0 || e >= E) {
        *bad = true;
        return -1;
    }
    return (int)e;
}

// step 1: counts of one chunk into LDS (s_cnt[w*E + e] per wave), returns via LDS
template <typename IdxT, int PERWAVE>
__device__ void chunk_wave_counts(const IdxT* idx, int64_t n, int E, int64_t chunk_base, int* s_cnt, bool* bad) {
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * E; i += 256) s_cnt[i] = 0;
    __syncthreads();
    for (int step = 0; step < PERWAVE / kWave; ++step) {
        const int64_t a = chunk_base + wave * PERWAVE + step * kWave + lane;
        const int e = load_expert(idx, a, n, E, bad);
        if (e >= 0) atomicAdd(&s_cnt[wave * E + e], 1);
    }
    __syncthreads();
}

// step 2 (one block): chunk_hist -> exclusive chunk bases (in place), hist, kept, offsets.  chunk_hist is
// [E, nchunks]: an expert's chunk counts lie side by side, so the lanes of a scanning wave read one line.
// A wave scans four experts at a time: 64 chunks per pass with a prefix sum over the wave, the carry
// runs across passes.
__device__ inline void scan_totals(int32_t* chunk_hist, int nchunks, int E, int C, int32_t* hist, int32_t* kept,
                            int32_t* offsets, int* s_tot) {
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int nwaves = blockDim.x >> 6;
    constexpr int U = 4;   // experts scanned together by a wave (their loads are issued back to back)
    constexpr int P = 2;   // passes of 64 chunks whose loads are issued together
    for (int e0 = wave * U; e0 < E; e0 += nwaves * U) {
        int carry[U];
#pragma unroll
        for (int u = 0; u < U; ++u) carry[u] = 0;
        for (int base = 0; base < nchunks; base += P * kWave) {
            int v[P][U];
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const int c = base + q * kWave + lane;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    v[q][u] = (c < nchunks && e0 + u < E) ? chunk_hist[(int64_t)(e0 + u) * nchunks + c] : 0;
            }
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const int c = base + q * kWave + lane;
                if (base + q * kWave >= nchunks) break;      // wave-uniform
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int incl = wave_inclusive_scan(v[q][u]);
                    if (c < nchunks && e0 + u < E) chunk_hist[(int64_t)(e0 + u) * nchunks + c] = carry[u] + incl - v[q][u];
                    carry[u] += __builtin_amdgcn_readlane(incl, kWave - 1);
                }
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (e0 + u < E) {
                    hist[e0 + u] = carry[u];
                    const int kp = carry[u] < C ? carry[u] : C;
                    kept[e0 + u] = kp;
                    s_tot[e0 + u] = kp;
                }
            }
        }
    }
    __syncthreads();
    // offsets = exclusive prefix sums of the kept counts: the first wave, 64 experts per step
    if (wave == 0) {
        int run = 0;
        for (int e0 = 0; e0 < E; e0 += kWave) {
            const int e = e0 + lane;
            const int kp = e < E ? s_tot[e] : 0;
            const int incl = wave_inclusive_scan(kp);
            if (e < E) offsets[e] = run + incl - kp;
            run += __builtin_amdgcn_readlane(incl, kWave - 1);
        }
        if (lane == 0) offsets[E] = run;
    }
    __syncthreads();
}

// step 3: ranks of one chunk.  s_cnt holds the per-wave counts of this chunk
// (from chunk_wave_counts); they are turned into per-wave running bases.
template <typename IdxT, int PERWAVE>
__device__ void chunk_rank_and_write(const IdxT* idx, int64_t n, int k, int E, int C, int64_t chunk_base,
                                     const int32_t* chunk_excl /* this chunk's entry of expert 0 */, int chunk_pitch,
                                     const int32_t* offsets, int* s_cnt, int32_t* slot, int32_t* token_map,
                                     int32_t* row_src, int32_t* row_of) {
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    // per-wave running base = chunk base + counts of the earlier waves
    for (int e = threadIdx.x; e < E; e += 256) {
        int run = chunk_excl[(int64_t)e * chunk_pitch];
        for (int w = 0; w < 4; ++w) {
            const int v = s_cnt[w * E + e];
            s_cnt[w * E + e] = run;
            run += v;
        }
    }
    __syncthreads();
    int* my_base = s_cnt + wave * E;
    const unsigned long long lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int step = 0; step < PERWAVE / kWave; ++step) {
        const int64_t a = chunk_base + wave * PERWAVE + step * kWave + lane;
        bool bad = false;
        const int e = load_expert(idx, a, n, E, &bad);
        int rank = -1;
        // the lanes of the same expert are those that agree with this one on every bit of its number (a turn of a loop per expert
        // took 4 us more where a step's 64 assignments name 40 of 64 experts: whole plans of 3600 assignments 10.7 -> 6.8 us, of 24576
        // 19.4 -> 14.9)
        unsigned long long same = __ballot(e >= 0);
        for (int b = 0; (E - 1) >> b; ++b) {
            const unsigned long long ones = __ballot(e >= 0 && ((e >> b) & 1));
            same &= ((e >> b) & 1) ? ones : ~ones;
        }
        if (e >= 0) {
            rank = my_base[e] + __popcll(same & lt_mask);
            asm volatile("" ::: "memory");        // every lane has read its base before a leader advances it
            if ((same & lt_mask) == 0) my_base[e] += __popcll(same);
        }
        if (a < n) {
            if (e >= 0 && rank < C) {
                const int row = offsets[e] + rank;
                slot[a] = rank;
                token_map[(int64_t)e * C + rank] = (int32_t)a;
                row_src[row] = (int32_t)a;
                row_of[a] = row;
            } else {
                slot[a] = -1;
                row_of[a] = -1;
            }
        }
    }
}

// Whole plan in one block (n <= kPlanSingle).  A chain of dependent steps, so what passes between them stays in registers
// (the expert ids) and LDS (counts, kept, offsets) instead of going through global memory, and waves and steps without
// assignments are skipped: 18 assignments to 64 experts take about 2 us behind the routing pass, 6.3 before.  NW: waves of
// the block.  s_all: (NW + 2) * E + 1 integers of LDS.
// s_idx: the ids again in LDS, or nullptr.
template <typename IdxT, int NW>
__device__ __forceinline__ void plan_single_block(const IdxT* idx, const int* s_idx, int64_t n, int k, int E, int C,
                                                  int32_t* hist, int32_t* kept, int32_t* offsets, int32_t* slot,
                                                  int32_t* token_map, int32_t* row_src, int32_t* row_of,
                                                  int64_t row_src_len, int32_t* status, int* s_all) {
    int* s_cnt = s_all;                    // [NW * E] counts, then running bases, per wave
    int* s_kept = s_all + NW * E;          // [E]
    int* s_off = s_all + (NW + 1) * E;     // [E + 1]
    constexpr int S = kPlanSingle / NW / kWave;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int ids[S];
    bool bad = false;
#pragma unroll
    for (int st = 0; st < S; ++st) {
        const int64_t a = wave * (S * kWave) + st * kWave + lane;
        ids[st] = -1;
        if (s_idx) {
            if (a < n) ids[st] = s_idx[a];
        } else {
            ids[st] = load_expert(idx, a, n, E, &bad);
        }
    }
    for (int i = threadIdx.x; i < NW * E; i += NW * 64) s_cnt[i] = 0;
    __syncthreads();
#pragma unroll
    for (int st = 0; st < S; ++st)
        if (ids[st] >= 0) atomicAdd(&s_cnt[wave * E + ids[st]], 1);
    const int any_bad = __syncthreads_or(bad ? 1 : 0);
    if (threadIdx.x == 0) status[0] = any_bad;
    for (int e = threadIdx.x; e < E; e += NW * 64) {
        int run = 0;                 // per-wave running base = counts of the earlier waves
        for (int w = 0; w < NW; ++w) {
            const int v = s_cnt[w * E + e];
            s_cnt[w * E + e] = run;
            run += v;
        }
        const int kp = run < C ? run : C;
        hist[e] = run;
        kept[e] = kp;
        s_kept[e] = kp;
    }
    __syncthreads();
    // offsets = exclusive prefix sums of the kept counts: the first wave, 64 experts per step
    if (wave == 0) {
        int run = 0;
        for (int e0 = 0; e0 < E; e0 += kWave) {
            const int e = e0 + lane;
            const int kp = e < E ? s_kept[e] : 0;
            const int incl = wave_inclusive_scan(kp);
            if (e < E) {
                s_off[e] = run + incl - kp;
                offsets[e] = run + incl - kp;
            }
            run += __builtin_amdgcn_readlane(incl, kWave - 1);
        }
        if (lane == 0) {
            s_off[E] = run;
            offsets[E] = run;
        }
    }
    __syncthreads();
    int* my_base = s_cnt + wave * E;
    const unsigned long long lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int st = 0; st < S; ++st) {
        const int64_t a = wave * (S * kWave) + st * kWave + lane;
        const int e = ids[st];
        // rank among the step's equal ids: the lanes that agree with this one on every bit of the id
        unsigned long long same = __ballot(e >= 0);
        if (same == 0 && wave * (S * kWave) + st * kWave >= n) break;       // wave-uniform
        for (int b = 0; (E - 1) >> b; ++b) {
            const unsigned long long ones = __ballot(e >= 0 && ((e >> b) & 1));
            same &= ((e >> b) & 1) ? ones : ~ones;
        }
        if (e >= 0) {
            const int rank = my_base[e] + __popcll(same & lt_mask);
            asm volatile("" ::: "memory");        // every lane has read its base before a leader advances it
            if ((same & lt_mask) == 0) my_base[e] += __popcll(same);
            if (rank < C) {
                const int row = s_off[e] + rank;
                slot[a] = rank;
                token_map[(int64_t)e * C + rank] = (int32_t)a;
                row_src[row] = (int32_t)a;
                row_of[a] = row;
            } else {
                slot[a] = -1;
                row_of[a] = -1;
            }
        } else if (a < n) {
            slot[a] = -1;
            row_of[a] = -1;
        }
    }
    const int ec = E * C;            // (below 2^31: checked on the host)
    for (int i = threadIdx.x; i < ec; i += NW * 64) {
        const int e = (int)((unsigned)i / (unsigned)C);
        if (i - e * C >= s_kept[e]) token_map[i] = -1;
    }
    for (int64_t i = s_off[E] + threadIdx.x; i < row_src_len; i += NW * 64) row_src[i] = -1;
}

}  // namespace ats
