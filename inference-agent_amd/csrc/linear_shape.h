// linear_shape.h — the workgroup shape of a batched linear call (linear_tile.hip): token blocks per
// tile, k groups, and the ways n_in is split over workgroups. Host code only.
#pragma once

#include <algorithm>
#include <cmath>

#include "linear_tile.h"

namespace ingot {

constexpr uint32_t kMaxSplits = 8, kMaxNtb = 4;

// Time (us) of a workgroup over 1024 elements of n_in: [k groups 4, 2, 1][token blocks of 32]. 0: no
// such kernel (F32: the weights' LDS leaves no room for 3 blocks on four k groups, their registers
// none for 4). And the bytes of 256 elements of a row.
struct TileCost {
    float walk[3][kMaxNtb + 1];
    float row256;
};
inline const TileCost& tile_cost(uint32_t type) {
    static constexpr TileCost q4_0{{{0, 2.8f, 4.2f, 5.7f, 0}, {0, 0, 6.7f, 8.0f, 9.8f}, {0, 0, 10.1f, 11.7f, 13.5f}}, 144};
    static constexpr TileCost q4_1{{{0, 3.7f, 5.0f, 6.4f, 0}, {0, 0, 8.2f, 9.5f, 10.9f}, {0, 0, 12.7f, 14.4f, 16.1f}}, 160};
    static constexpr TileCost q8_0{{{0, 3.8f, 5.6f, 7.0f, 0}, {0, 0, 8.3f, 10.1f, 12.2f}, {0, 0, 13.1f, 14.8f, 16.5f}}, 272};
    static constexpr TileCost q6_k{{{0, 5.5f, 6.8f, 9.3f, 0}, {0, 0, 11.5f, 12.3f, 15.2f}, {0, 0, 17.9f, 19.8f, 25.0f}}, 210};
    static constexpr TileCost f16{{{0, 3.5f, 5.3f, 7.2f, 0}, {0, 0, 7.5f, 9.3f, 11.4f}, {0, 0, 11.6f, 13.8f, 15.5f}}, 512};
    static constexpr TileCost bf16{{{0, 3.7f, 5.7f, 7.5f, 0}, {0, 0, 8.0f, 10.0f, 12.1f}, {0, 0, 12.4f, 14.6f, 16.0f}}, 512};
    static constexpr TileCost f32{{{0, 5.1f, 7.0f, 0, 0}, {0, 0, 10.6f, 12.6f, 0}, {0, 0, 18.2f, 20.8f, 0}}, 1024};
    switch (type) {
        case 0:  return f32;
        case 1:  return f16;
        case 3:  return q4_1;
        case 8:  return q8_0;
        case 14: return q6_k;
        case 30: return bf16;
        default: return q4_0;
    }
}

constexpr int tile_kg_row(uint32_t kg) { return kg == 4 ? 0 : kg == 2 ? 1 : 2; }

inline bool tile_fits(uint32_t type, uint32_t n_in, uint32_t kg, uint32_t ntb) {
    if (tile_cost(type).walk[tile_kg_row(kg)][ntb] == 0) return false;
    return ntb <= 2 || uint64_t(128) * ntb * n_in < 0x80000000ull;  // 32-bit offsets into a tile's x
}

inline uint64_t tile_count(uint32_t n_out, uint32_t n_tok, const TileShape& s) {
    const uint32_t tr = tile_rows(s.kg), nb = (n_tok + 31) / 32;
    return uint64_t((n_out + tr - 1) / tr) * ((nb + s.ntb - 1) / s.ntb);
}

// Estimated time (us) of a shape on n_out rows: the launch; rounds of 256 workgroups, each a fixed part
// and the longest share of n_in (whole units), slower the more W and x the workgroups read from the
// L2s, and hardly faster than the eight XCDs fetch their shares of x (6.2 TB/s) and W (3.6 TB/s);
// the output's stores; and where n_in is split the partial tiles' stores and the last workgroup's
// reading them. Fitted to 133 thousand timings, over half with weights that no cache holds, as a
// model's are: seven types, 24 sets of matrices (512 .. 14336 columns, 512 .. 28672 rows), 2 to 1024
// tokens, every shape. Against the best shape timed, the one it picks is 0.8% slower in the mean and 5%
// in the worst twentieth (one matrix; 0.1% and 0 q/k/v, 0.4% and 4% gate/up). The former rule, one
// table in proportion for all types, took 2.4% more over single matrices and 5 to 6% over sets.
inline float tile_us(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, const TileShape& s) {
    const TileCost& c = tile_cost(type);
    const uint32_t tiles_m = ((n_tok + 31) / 32 + s.ntb - 1) / s.ntb, rows = tile_rows(s.kg);
    const float splits = float(s.splits), wgs = float(tile_count(n_out, n_tok, s)) * splits;
    const float rounds = float(uint64_t(wgs + 255.f) / 256);
    const uint32_t share = (tile_units(type, n_in, s.kg) + s.splits - 1) / s.splits * tile_unit(type) * s.kg;
    const float k = float(share) / 1024.f, row = c.row256 / 256.f;
    const float reads = (float(rows) * row + 128.f * float(s.ntb)) / 256.f;  // of an element of n_in, 256 bytes
    const float walk = rounds * (2.8f + k * c.walk[tile_kg_row(s.kg)][s.ntb]) + 0.4f * k * reads * wgs / 256.f;
    // An XCD takes a contiguous run of (row tile, token tile, split) ids: the part of x and of W in it.
    const float run = float(uint64_t(wgs + 7.f) / 8), turns = run / (float(tiles_m) * splits);
    const float x = std::min(1.f, turns) * float(n_tok) * 4.f;
    const float w = (run >= splits ? std::max(1.f, turns) : run / splits) * float(rows) * row;
    const float fetch = 8e-7f * float(n_in) * (1.3f * x + 2.2f * w);
    const float w2 = walk * walk, f2 = fetch * fetch, part = float(tile_bytes(s));
    const float t = 2.9f + std::sqrt(std::sqrt(w2 * w2 + f2 * f2)) + 2.5e-7f * wgs * part;
    if (s.splits == 1) return t;
    return t + 1.f + 0.3f * splits * part / 32768.f + 6e-8f * wgs * part;
}

// The tile height of least estimated time; it does not change the order of an output's sum.
inline TileShape tile_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t kg, uint32_t splits,
                            float& us) {
    TileShape best{0, kg, splits};
    for (uint32_t ntb = 1; ntb <= kMaxNtb; ntb++) {
        if (!tile_fits(type, n_in, kg, ntb)) continue;
        const float u = tile_us(type, n_in, n_out, n_tok, TileShape{ntb, kg, splits});
        if (best.ntb == 0 || u < us) { best.ntb = ntb; us = u; }
    }
    return best;
}

// The k groups of a matrix in a call that is not split. They order each output's sum, so they depend
// on the matrix and n_tok alone, not on what shares the launch: ingot_proj equals ingot_linear bit
// for bit. They are the best for the rows that usually run together. A matrix wider than n_in is half
// of a gate/up pair. One up to n_in is a part of q/k/v, 1.25 (70B, 8 KV heads) to 3 n_in rows (no
// grouped heads): 1.6 is taken up to 4096, 2.2 above, where both kinds stay within 2% of the better
// choice in the mean (with 1.6 throughout 3 x 5120 x 5120 lost 11%, with 2.2 6144 x 4096 8%). Except
// that with n_in above 5120 and 1.3 to 5 times its rows it is a down projection and runs alone.
// (2 x 4096 x 1024 Q4_0 at 288 tokens: 25.2 us on four k groups, 17.5 on two; 2 x 14336 x 4096 F16 at
// 70: 78.0 and 59.9.)
inline uint32_t unsplit_k_groups(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok) {
    const uint64_t in = n_in, out = n_out;
    const bool wide = 10 * out > 13 * in, alone = in > 5120 && 4 * out <= 3 * in && 5 * out > in;
    const uint64_t together = wide ? 2 * out : alone ? out : in * (in <= 4096 ? 8 : 11) / 5;
    const uint32_t rows = uint32_t(std::min<uint64_t>(together, 0x7fffffffu));
    uint32_t best = 4;
    float t = 0;
    for (uint32_t kg = 4; kg >= 1; kg /= 2) {
        float u = 0;
        tile_shape(type, n_in, rows, n_tok, kg, 1, u);
        if (kg == 4 || u < t) { best = kg; t = u; }
    }
    return best;
}

// The shape of matrices of n_out rows together, on kg k groups, not split.
inline TileShape unsplit_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t kg) {
    float us = 0;
    return tile_shape(type, n_in, n_out, n_tok, kg, 1, us);
}

// The shape of a call on one matrix whose workspace lets n_in be split: of all shapes, the one of
// least estimated time (wo 3072 x 3072 Q4_0 at 13 tokens: 13.1 us unsplit, 9.1 in five; down
// 8192 x 3072 at 157: 64.8 and 27.5 us); a split costs up to 2% less than estimated up to 128 tokens
// (Q4_0 3072 x 3072 at 128: 14.2 us in two, 14.5 unsplit) and more beyond, where the last workgroup of a
// large tile also adds to out (wo at 512: 30.8 unsplit, 31.9 in two; of 1862 such calls 33 were more than
// 3% slower than the former rule's choice with 1.06 here, 42 with 1.03). A requested count takes two
// k groups, or one where n_in has too few units of two.
inline TileShape linear_shape(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t requested,
                              size_t workspace_bytes) {
    const uint32_t cap = std::min(kMaxSplits, std::max(1u, n_in / 256));  // at least 256 elements a split
    if (requested == 1 || cap == 1 || workspace_bytes <= kLinearCounterBytes)
        return unsplit_shape(type, n_in, n_out, n_tok, unsplit_k_groups(type, n_in, n_out, n_tok));
    requested = std::min(requested, cap);
    TileShape best{};
    float t = 0;
    for (uint32_t kg = 4; kg >= 1; kg /= 2) {
        const uint32_t units = tile_units(type, n_in, kg);
        if (requested > 1 && kg != (tile_units(type, n_in, 2) >= requested ? 2u : 1u)) continue;
        const uint32_t last = requested > 1 ? requested : std::min(cap, units);
        for (uint32_t splits = std::max(requested, 1u); splits <= last; splits++)
            for (uint32_t ntb = 1; ntb <= kMaxNtb; ntb++) {
                const TileShape s{ntb, kg, splits};
                if (!tile_fits(type, n_in, kg, ntb)) continue;
                const uint64_t tiles = tile_count(n_out, n_tok, s);
                if (splits > 1 && (tiles > kLinearMaxTiles ||
                                   kLinearCounterBytes + tiles * splits * tile_bytes(s) > workspace_bytes)) continue;
                const float u = tile_us(type, n_in, n_out, n_tok, s) * (splits == 1 ? 1.f : n_tok <= 128 ? 0.98f : 1.06f);
                if (best.ntb == 0 || u < t) { best = s; t = u; }
            }
    }
    // (no room for the requested splits)
    return best.ntb ? best : unsplit_shape(type, n_in, n_out, n_tok, unsplit_k_groups(type, n_in, n_out, n_tok));
}

}  // namespace ingot
