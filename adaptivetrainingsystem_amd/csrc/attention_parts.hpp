// Which query tiles of a head a workgroup of the causal attention kernels takes.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace ats {

constexpr int kAttnMaxTiles = 32, kAttnMaxParts = 16;

// count workgroups per head; bit t of tiles[p]: part p takes tile t.  count == 0: part p takes tile n - 1 - p and tile p.
struct AttnParts {
    int count;
    uint32_t tiles[kAttnMaxParts];
};

// A part's work is counted in key tiles, kTileStart more for each query tile (its first loads, its epilogue: 1.0 us a key tile and
// 4-6 of them measured).  The parts of a launch run one or two at a time on a compute unit, two of them 1.25 times as long as one by
// itself (1.95 against 1.08 us a key tile were they in step all the way; the factor that chose best among 2.5 .. 4 quarters a pair).  Pairs are even, but
// as many as the tiles make: 96 heads of 14 tiles are 84 pairs of 30 key tiles on an XCD's 32 units, three on some and two on others.
// Five parts of 42 (28 + 14, 26 + 16, 24 + 18, 22 + 20, the rest) are two on nearly every unit: 3 x 1777 positions, 32 heads of 128,
// 120 -> 103 us (with the queries' rotation 145 -> 129; the layer 505 -> 500, its products run a little slower behind it: board
// power), 1 x 4737 of 32 heads of 64 185 -> 130 (the layer 314 -> 254).  70 random shapes of 1-8 sequences of 129-8192 positions: the forward takes
// 11 % less time on average than in pairs (0.76 .. 1.05 of it), the backward with its queries in one range 10 % (0.69 .. 1.03).  A twentieth
// is what the estimate has to promise; more than 32 tiles of a head keep to pairs, whose number is then large.
//
// work(t): key tiles that query tile t sees (not falling with t); n_heads heads share `cus` compute units, each of which runs
// `two` or one workgroup at a time.  *estimate: time of the fullest compute unit in quarters of a lone workgroup's key tile.
template <typename F>
inline AttnParts attn_parts(int n_tiles, int64_t n_heads, int cus, bool two, F work, int64_t* estimate = nullptr) {
    constexpr int kTileStart = 6;
    AttnParts best{};
    auto cost = [&](int parts, int64_t most) {
        const int64_t per_cu = (n_heads * parts + cus - 1) / cus;
        return most * (two ? 5 * (per_cu / 2) + 4 * (per_cu % 2) : 4 * per_cu);
    };
    int most = n_tiles % 2 ? work(n_tiles / 2) + kTileStart : 0;
    for (int p = 0; p < n_tiles / 2; ++p) most = std::max(most, work(p) + work(n_tiles - 1 - p) + 2 * kTileStart);
    if (estimate) *estimate = cost((n_tiles + 1) / 2, most);
    if (n_tiles < 2 || n_tiles > kAttnMaxTiles || n_heads < 1) return best;
    int64_t least = cost((n_tiles + 1) / 2, most) * 19 / 20;
    int w[kAttnMaxTiles], total = 0;
    for (int t = 0; t < n_tiles; ++t) total += w[t] = work(t) + kTileStart;
    // first fit, the longest tile first: whether `parts` parts of that much room hold all tiles
    auto fit = [&](int parts, int room, AttnParts* a) {
        *a = AttnParts{};
        a->count = parts;
        int left[kAttnMaxParts];
        for (int p = 0; p < parts; ++p) left[p] = room;
        for (int t = n_tiles - 1; t >= 0; --t) {
            int p = 0;
            while (p < parts && left[p] < w[t]) ++p;
            if (p == parts) return false;
            left[p] -= w[t];
            a->tiles[p] |= 1u << t;
        }
        return true;
    };
    for (int parts = std::min(n_tiles, kAttnMaxParts); parts >= 1; --parts) {
        // the least room between what a part needs at least and the most that promises anything, which lie a few key tiles apart where
        // all keys are new (0.3-3 us a call); by halves where tiles are longer (with a million cached keys they are tens of thousands
        // of key tiles, and trying each room took 6 ms of every call)
        int lo = std::max(w[n_tiles - 1], (total + parts - 1) / parts);
        int hi = (int)std::min<int64_t>((least - 1) / cost(parts, 1), total);
        AttnParts a;
        if (hi - lo < 64) {
            while (lo <= hi && !fit(parts, lo, &a)) ++lo;
            if (lo > hi) continue;
        } else {
            if (!fit(parts, hi, &a)) continue;
            while (lo < hi) {
                const int mid = lo + (hi - lo) / 2;
                AttnParts b;
                if (fit(parts, mid, &b)) hi = mid, a = b;
                else lo = mid + 1;
            }
        }
        if (a.tiles[parts - 1]) {      // (fewer parts hold them as well: a later turn)
            least = cost(parts, lo);
            best = a;
            if (estimate) *estimate = least;
        }
    }
    return best;
}

}  // namespace ats
