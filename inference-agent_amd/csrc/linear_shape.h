// linear_shape.h — the workgroup shape of a batched linear call (linear_tile.hip): token blocks per
// tile, k groups, and the ways n_in is split over workgroups. Host code only.
#pragma once

#include <algorithm>

#include "linear_tile.h"

namespace ingot {

constexpr uint32_t kTypeF32 = 0, kTypeQ6_K = 14;  // GGUF type ids

// Measured time of one workgroup over 3072 elements of n_in beside its fixed part of ~4 us (us):
// [k groups 4, 2, 1][token blocks of 32], of Q4_0 (the other types are near it in proportion) and of
// Q6_K, whose dequantization weighs more against the token blocks. 0: no such kernel.
constexpr uint32_t kMaxSplits = 8, kMaxNtb = 4;
inline float tile_walk_us(uint32_t type, uint32_t kg, uint32_t ntb) {
    constexpr float t[2][3][kMaxNtb + 1] = {{{0, 9, 13, 19, 0}, {0, 0, 20, 25, 31}, {0, 0, 30, 40, 50}},
                                            {{0, 18, 24, 30, 0}, {0, 0, 40, 45, 48}, {0, 0, 60, 68, 77}}};
    return t[type == kTypeQ6_K][kg == 4 ? 0 : kg == 2 ? 1 : 2][ntb];
}

inline bool tile_fits(uint32_t type, uint32_t n_in, uint32_t kg, uint32_t ntb) {
    if (tile_walk_us(type, kg, ntb) == 0) return false;
    // F32: the weights' LDS leaves no room for 3 blocks on four k groups, their registers none for 4
    // (they spill: gate/up at 512 tokens 180.7 us).
    if (type == kTypeF32 && (ntb == 4 || (kg == 4 && ntb == 3))) return false;
    return ntb <= 2 || uint64_t(128) * ntb * n_in < 0x80000000ull;  // 32-bit offsets into a tile's x
}

// Estimated time (us) of a shape: rounds of 256 workgroups, each the longest share of n_in (whole
// units), then the tail of a split: the last workgroup of a tile reads every split's partial tile
// (~32 KB a us).
inline float tile_us(uint32_t type, uint32_t n_in, uint64_t tiles, const TileShape& s) {
    const float rounds = float((tiles * s.splits + 255) / 256);
    const uint32_t share = (tile_units(type, n_in, s.kg) + s.splits - 1) / s.splits * tile_unit(type) * s.kg;
    const float t = rounds * (4.f + tile_walk_us(type, s.kg, s.ntb) * float(share) / 3072.f);
    return s.splits == 1 ? t : t + 3.f + float(s.splits * tile_bytes(s)) / 32768.f;
}

inline uint64_t tile_count(uint32_t n_out, uint32_t n_tok, const TileShape& s) {
    const uint32_t tr = tile_rows(s.kg), nb = (n_tok + 31) / 32;
    return uint64_t((n_out + tr - 1) / tr) * ((nb + s.ntb - 1) / s.ntb);
}

// A call that is not split: the number of k groups depends on n_tok and on which side of 4096 rows
// each matrix is, so that every output is summed in the same order whatever else shares the launch
// (ingot_proj equals ingot_linear bit for bit; it launches matrices of both sides apart). The tile
// height, which does not change the order, is the one that takes least time for n_out rows.
// Measured on Q4_0 rows of 3072 (four, two, one k groups, us): gate/up of 2 x 8192 rows at 70
// tokens 27.7 / 31 / 38, at 157 49.5 / 37.1 / 38.9, at 512 143 / 88 / 67; q/k/v of 3072 + 2 x 1024
// rows at 157 tokens 17.4 / 24.3 / 33.7, at 256 23.2 / 26.2 / 34.7, at 389 41.4 / 29.8 / 34.7, at
// 512 44 / 32.8 / 35.2.
constexpr uint32_t kNarrowRows = 4096;
inline TileShape unsplit_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, bool narrow) {
    const uint32_t nb = (n_tok + 31) / 32;
    TileShape best{0, narrow ? (nb <= 9 ? 4u : 2u) : nb <= 3 ? 4u : nb <= 9 ? 2u : 1u, 1};
    float t = 0;
    for (uint32_t ntb = 1; ntb <= kMaxNtb; ntb++) {
        if (!tile_fits(type, n_in, best.kg, ntb)) continue;
        const TileShape s{ntb, best.kg, 1};
        const float u = tile_us(type, n_in, tile_count(n_out, n_tok, s), s);
        if (best.ntb == 0 || u < t) { best.ntb = ntb; t = u; }
    }
    return best;
}

// The shape of a call on one matrix whose workspace lets n_in be split: of all shapes, the one of
// least estimated time (wo 3072 x 3072 Q4_0 at 13 tokens: 13.1 us unsplit, 9.1 in five; down
// 8192 x 3072 at 157: 64.8 and 27.5 us). Up to 128 tokens it always splits (within 2% of
// unsplit at 128). A requested count takes two k groups, or one where n_in has too few units of two.
inline TileShape linear_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t requested,
                              size_t workspace_bytes) {
    const TileShape un = unsplit_shape(type, n_in, n_out, n_tok, n_out <= kNarrowRows);
    const uint32_t cap = std::min(kMaxSplits, std::max(1u, n_in / 256));  // at least 256 elements a split
    if (requested == 1 || cap == 1 || workspace_bytes <= kLinearCounterBytes) return un;
    requested = std::min(requested, cap);
    TileShape best = un;
    float t = tile_us(type, n_in, tile_count(n_out, n_tok, un), un);
    bool split = false;
    for (uint32_t kg = 4; kg >= 1; kg /= 2) {
        const uint32_t units = tile_units(type, n_in, kg);
        if (requested > 1 && kg != (tile_units(type, n_in, 2) >= requested ? 2u : 1u)) continue;
        for (uint32_t ntb = 1; ntb <= kMaxNtb; ntb++) {
            if (!tile_fits(type, n_in, kg, ntb)) continue;
            const uint32_t last = requested > 1 ? requested : std::min(cap, units);
            for (uint32_t splits = std::max(requested, 1u); splits <= last; splits++) {
                const TileShape s{ntb, kg, splits};
                const uint64_t tiles = tile_count(n_out, n_tok, s);
                const bool fits = splits == 1 ||
                    (tiles <= kLinearMaxTiles && kLinearCounterBytes + tiles * splits * tile_bytes(s) <= workspace_bytes);
                const float u = tile_us(type, n_in, tiles, s);
                const bool must = (requested > 1 || n_tok <= 128) && splits > 1;  // a split is wanted
                if (fits && ((must && !split) || (must == split && u < t))) {
                    best = s;
                    t = u;
                    split = must;
                }
            }
        }
    }
    return best;
}

}  // namespace ingot
