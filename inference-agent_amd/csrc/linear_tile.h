// linear_tile.h — the launcher of the batched linear kernel (linear_tile.hip), one object per
// weight type.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ingot {

// Linear layer workspace: split-K completion counters (one 64-byte line per output tile, for up
// to kLinearMaxTiles tiles), then the partial tiles.
constexpr size_t kLinearCounterBytes = 16384;
constexpr uint32_t kLinearMaxTiles = 256;

// Shape of a call's workgroups: NTB token blocks of 32 per tile (1..4), KG k groups among the
// eight waves (1, 2 or 4: a tile has 256 / KG rows), and the ways n_in is split over workgroups.
struct TileShape {
    uint32_t ntb, kg, splits;
};

struct TileCall {
    const uint8_t* W[3];
    float* out[3];
    uint32_t n_out[3];
    uint32_t n_mats;
    const float* x;
    uint32_t n_in, n_tok;
    bool accumulate;
    bool pair;  // W = (gate, up): out[0] = silu(gate) * up
    TileShape shape;
    void* workspace;  // counters, then partial tiles (shape.splits > 1)
    hipStream_t stream;
    bool spread = false;  // the order of the sums is free (see tile_spread)
    uint32_t row0 = 0, rows = ~0u;  // the rows of each matrix to compute (out keeps its n_out columns)
};

// Rows per tile, k elements per stage and bytes of one partial tile of a shape.
constexpr uint32_t tile_rows(uint32_t kg) { return 256 / kg; }
// A stage: 64-element steps of each k group (two where one k group fits the LDS), and elements.
constexpr uint32_t tile_cols(uint32_t kg) { return kg == 1 ? 2 : 1; }
constexpr uint32_t tile_stage(uint32_t kg) { return 64 * kg * tile_cols(kg); }
// A k group's share of n_in is a multiple of this many elements (whole Q6_K blocks).
constexpr uint32_t tile_unit(int type) { return type == 14 ? 256 : 64; }
// n_in in units of every k group's share of that many elements; a call is split over whole units.
constexpr uint32_t tile_units(int type, uint32_t n_in, uint32_t kg) {
    const uint64_t u = uint64_t(tile_unit(type)) * kg;
    return uint32_t((n_in + u - 1) / u);
}
// The two x buffers.
constexpr size_t tile_x_lds(uint32_t ntb, uint32_t kg) { return size_t(2) * 32 * ntb * tile_stage(kg) * 2; }
// LDS of a workgroup: the x buffers and the waves' weights, reused by the reduction over the k
// groups and the silu exchange (16 floats per lane, token block and wave).
constexpr size_t tile_lds(uint32_t ntb, uint32_t kg, size_t w) {
    const size_t x = tile_x_lds(ntb, kg) + w;
    const size_t red = size_t(kg - 1) * (8 / kg) * ntb * 4096, silu = size_t(4 / kg) * ntb * 4096;
    return x > red ? (x > silu ? x : silu) : (red > silu ? red : silu);
}
constexpr size_t tile_bytes(const TileShape& s) { return size_t(tile_rows(s.kg)) * s.ntb * 32 * 4; }

// Do the token tiles of a call start their walks of n_in apart? It pays where what one tile has read stays
// in the XCD's 4 MB of L2 until the last has (w: bytes of the rows, an eighth on each XCD; x: bytes of x),
// measured on two k groups (with weights from HBM, 2 to 1024 tokens, 0.90 to 1.20x of in step): F16 and BF16
// 1.047x in the mean up to w = 20 MB and x = 9 MB (3072 x 3072: 256 tokens 24.0 -> 21.4 us, 512 34.4 ->
// 28.7; the worst, 1024 x 4096 at 700, 18.2 -> 20.3), 0.91 to 0.96x with w = 33 MB or with w = 17 MB and x from 9.4 MB on; Q8_0, Q4_0 and Q4_1 1.02x,
// Q6_K 1.00x. On one k group 256 rows share a walk and lose more than they gain from 2 MB on (0.98x,
// 0.92x, 0.89x at 2, 4 and 7 MB an XCD); calls on four have few token tiles.
inline bool tile_spread(const TileShape& s, uint64_t w, uint64_t x) {
    return s.kg == 2 && w <= 20000000 && x <= 9000000;
}
// First of part i's share where n things are spread evenly over `parts`, the first n % parts parts one
// longer: the token blocks of a token tile, the k units of a split. (i * n / parts would pass 32 bits
// from 2.1 million tokens of one-block tiles, 4.2 million of four-block tiles on.)
constexpr uint32_t tile_share0(uint32_t i, uint32_t n, uint32_t parts) {
    const uint32_t longer = n % parts;
    return i * (n / parts) + (i < longer ? i : longer);
}

// 0, -1 (grid too large or a bad shape) or -4 (launch failed). T: the GGUF type id.
template <int T> int launch_tile(const TileCall& c);

}  // namespace ingot
