// linear_tile.hip — out (+)= W·x for several tokens over one GGUF weight type, for gfx950.
// Compiled once per type (INGOT_TILE_TYPE, a type id of linear_formats.h).
//
// Like the Metal path (to_half + matmul_tiles, src/metal_backend.mm:385-392, shaders/
// kernels.metal:779-850) x and the dequantized weights are rounded to f16 and products accumulate
// in f32, on v_mfma_f32_32x32x16_f16 with the weights as the A operand, so that a lane ends with
// four consecutive rows of one token: 16 contiguous bytes of out.
//
// A workgroup is eight waves over 32 * NTB tokens and 256 / KG rows: KG k groups of 8 / KG waves,
// each wave on 32 rows and a contiguous share of n_in, the shares summed through LDS in order. A
// wave's weights are dequantized once for all tokens of the tile, in registers, straight into the
// MFMA operand (a lane owns one 32-element block of a row per step); only x, shared by the waves,
// is kept in LDS as f16. Few tokens take four k groups: narrow tiles of rows fill the chip
// without splitting n_in over workgroups.
//
// What bounds it: a few tokens, the latency of the chain launch - first loads - walk - tail (13
// tokens, 5120 x 3072 Q8_0: 57.7 us on one-k-group tiles of 256 rows, 18.6 here); a full chunk, the
// x stream and the dequantization that the MFMAs wait for (512 tokens, gate/up of 3072 -> 2 x 8192
// Q8_0: 124.6 -> 77 us, Q4_0 80.3 -> 65: 790 TFLOP/s, matrix cores busy 34% of the counted cycles).
// Token tiles that walk the same rows in step all wait for HBM at every stage: a square of 3072 in F16
// with weights that no cache holds took 32.4 us at 512 tokens, from the cache 25.5 (the kernel before
// this one 27.5); with their walks spread over the rows (tile_spread) 27.2. Measured
// on the way there, 512 tokens of Q4_0 gate/up: weights read by each lane straight from memory
// made the L1 fetch every line 5 times over (7.5 M line reads a launch, 5.3 M with whole rows
// through LDS); a branch around the dequantization of a ragged end kept the compiler from
// interleaving MFMAs with it (67 M wave-cycles, 52 M without); starting the token tiles at
// different stages changed nothing there (rows of that size do not stay in the L2).
#include <algorithm>
#include <type_traits>

#include "linear_formats.h"
#include "linear_tile.h"

namespace ingot {

namespace {

constexpr int kScDevice = 16;  // buffer cache-policy bits: sc1 = device scope
constexpr uint32_t kOob = 0x80000000u;  // an offset past every descriptor's range: loads zeros

// Operand e (elements 8e..8e+7) of a lane's column as f16; with kFragSwap13 the order within each
// four elements is 0,2,1,3. Weights are rounded to f16 from their exact f32 value. off: the
// column's byte offset (its place in the window). keep: ~0, or 0 for a block column past the end
// (its scale is cleared, so that it counts as zero).
template <int T>
__device__ __forceinline__ half8 col_frag(const uint32_t (&w)[Col<T>::ndw], uint32_t off, uint32_t c, uint32_t keep, int e) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    half8 o;
    if constexpr (T == kF16) {
        o = __builtin_bit_cast(half8, u32x4{w[4 * e], w[4 * e + 1], w[4 * e + 2], w[4 * e + 3]});
    } else if constexpr (T == kBF16) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o[2 * i] = _Float16(__uint_as_float(w[4 * e + i] << 16));
            o[2 * i + 1] = _Float16(__uint_as_float(w[4 * e + i] & 0xFFFF0000u));
        }
    } else if constexpr (T == kF32) {
#pragma unroll
        for (int i = 0; i < 8; i++) o[i] = _Float16(__uint_as_float(w[8 * e + i]));
    } else if constexpr (T == kQ4_0 || T == kQ8_0) {
        // Packed f16, two elements two bytes apart per word. Q4_0: a low nibble n becomes the half
        // 1024 + n (bits 0x6400 | n), minus 1032 gives n - 8; a high one becomes 1024 + 16 n, times
        // 1/16 minus 72 (one fma) the same; both exact. Times d rounds once: the f32 value
        // d * (n - 8) rounded to half. Q8_0: q ^ 0x80 = q + 128 becomes 1024 + q + 128, minus 1152
        // gives q, times d. The block starts at byte 0 or 2 of its window: v_perm picks the
        // scale (twice) and the quants at either place.
        const bool odd = (off & 2) != 0;
        const uint32_t qsel = odd ? 0x07060504u : 0x05040302u, dsel = odd ? 0x03020302u : 0x01000100u;
        const h2 dd = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0, w[0], dsel) & keep);
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int i = T == kQ4_0 ? 2 * (e & 1) + p : 2 * e + p;  // dword of the block's quants
            uint32_t q = __builtin_amdgcn_perm(w[i + 1], w[i], qsel);
            if constexpr (T == kQ8_0) q ^= 0x80808080u;
            const bool hi = T == kQ4_0 && e >= 2;  // elements 16..31 are the high nibbles
            const uint32_t mask = T == kQ8_0 ? 0x00FF00FFu : hi ? 0x00F000F0u : 0x000F000Fu;
            const _Float16 z = T == kQ8_0 ? _Float16(-1152.f) : hi ? _Float16(-72.f) : _Float16(-1032.f);
            const h2 zz = {z, z}, r16 = {_Float16(0.0625f), _Float16(0.0625f)};
            h2 a = __builtin_bit_cast(h2, and_or(q, mask, 0x64006400u));
            h2 b = __builtin_bit_cast(h2, and_or(q >> 8, mask, 0x64006400u));
            a = (hi ? __builtin_elementwise_fma(a, r16, zz) : a + zz) * dd;
            b = (hi ? __builtin_elementwise_fma(b, r16, zz) : b + zz) * dd;
            o[4 * p] = a[0];
            o[4 * p + 1] = a[1];
            o[4 * p + 2] = b[0];
            o[4 * p + 3] = b[1];
        }
    } else if constexpr (T == kQ4_1) {
        const float d = f16_bits(w[0] & keep & 0xFFFF), m = f16_bits((w[0] & keep) >> 16);
#pragma unroll
        for (int i = 0; i < 8; i++)
            o[i] = _Float16(d * float((w[1 + 2 * (e & 1) + i / 4] >> (8 * (i & 3) + 4 * (e >> 1))) & 0xF) + m);
    } else {  // Q6_K
        // sc*(q - 32) as fma(sc, q, -32*sc): -32*sc is exact, the fma rounds the exact value once.
        const uint32_t h = (c >> 2) & 1, g = c & 3;
        const uint32_t sl = (off + 64 * h + 32 * (g & 1)) & 3, sh = (off + 128 + 32 * h) & 3;
        const uint32_t nib = g >= 2 ? 4 : 0, hb = 2 * g;
        const float d = f16_bits(((w[19] & keep) >> (8 * ((off + 208) & 3))) & 0xFFFF);
        const uint32_t scw = w[18] >> (8 * ((off + 192 + 8 * h + 2 * g) & 3));
        const float sc = d * float(int8_t((e < 2 ? scw : scw >> 8) & 0xFF)), z = -32.f * sc;
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int i = 2 * e + p;
            const uint32_t ql = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sl);
            const uint32_t qh = __builtin_amdgcn_alignbyte(w[9 + i + 1], w[9 + i], sh);
            const uint32_t q = ((ql >> nib) & 0x0F0F0F0Fu) | (((qh >> hb) & 0x03030303u) << 4);
#pragma unroll
            for (int b = 0; b < 4; b++) o[4 * p + b] = _Float16(__builtin_fmaf(sc, float((q >> (8 * b)) & 0xFF), z));
        }
    }
    return o;
}

// A wave's weights go through LDS (its own region, no barrier): a W stage is WK elements of its 32
// rows, loaded in whole 16-byte chunks a stage ahead in registers (consecutive lanes take
// consecutive chunks of a row, so each cache line is fetched once), CH chunks from the 16-byte
// boundary at or below the row's piece, stored at a pitch that keeps the column reads at most
// two-way conflicted.
template <int T> struct WStage;
template <> struct WStage<kF32>  { static constexpr uint32_t WK = 64,  CH = 16, pitch = 272; };
template <> struct WStage<kF16>  { static constexpr uint32_t WK = 64,  CH = 8,  pitch = 144; };
template <> struct WStage<kBF16> { static constexpr uint32_t WK = 64,  CH = 8,  pitch = 144; };
template <> struct WStage<kQ8_0> { static constexpr uint32_t WK = 128, CH = 10, pitch = 176; };
template <> struct WStage<kQ4_0> { static constexpr uint32_t WK = 256, CH = 10, pitch = 176; };
template <> struct WStage<kQ4_1> { static constexpr uint32_t WK = 256, CH = 12, pitch = 208; };
template <> struct WStage<kQ6_K> { static constexpr uint32_t WK = 256, CH = 14, pitch = 240; };

// On one k group the 16-bit types take stages of 128 elements, whole 256-byte pieces of a row, which
// come faster from HBM (F16 and BF16 weights that no cache holds, mean of 19 token counts by 10 sets of
// matrices: 1.05 to 1.08x); on more, where a wave's share is short, the longer first load costs more
// (0.91 to 0.99x).
struct WStage128 { static constexpr uint32_t WK = 128, CH = 16, pitch = 272; };
template <int T, int KG>
using Staged = std::conditional_t<KG == 1 && (T == kF16 || T == kBF16), WStage128, WStage<T>>;

// The window of the column at byte `off` of a row in LDS (col_load's dwords).
template <int T>
__device__ __forceinline__ void col_read(const uint8_t* row, uint32_t off, uint32_t c, uint32_t (&w)[Col<T>::ndw]) {
    auto dw = [&](uint32_t o) { return *reinterpret_cast<const uint32_t*>(row + o); };
    if constexpr (T == kQ6_K) {
        const uint32_t h = (c >> 2) & 1, g = c & 3;
        const uint32_t pl = (off + 64 * h + 32 * (g & 1)) & ~3u, ph = (off + 128 + 32 * h) & ~3u;
#pragma unroll
        for (int i = 0; i < 9; i++) { w[i] = dw(pl + 4 * i); w[9 + i] = dw(ph + 4 * i); }
        w[18] = dw((off + 192 + 8 * h + 2 * g) & ~3u);
        w[19] = dw((off + 208) & ~3u);
    } else if constexpr (T == kF16 || T == kBF16 || T == kF32) {
#pragma unroll
        for (int i = 0; i < Col<T>::ndw / 4; i++) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(row + off + 16 * i);
            for (int e = 0; e < 4; e++) w[4 * i + e] = v[e];
        }
    } else {
#pragma unroll
        for (int i = 0; i < Col<T>::ndw; i++) w[i] = dw((off & ~3u) + 4 * i);
    }
}

struct TileArgs {
    const uint8_t* W[3];
    float* out[3];
    uint32_t n_out[3];     // rows [row0, n_out[m]) of matrix m, whose out has ld[m] columns
    uint32_t ld[3], row0;
    uint32_t tile_end[2];  // row tiles of matrix m: [tile_end[m-1], tile_end[m])
    const float* x;
    uint32_t n_in, n_tok, row_bytes, accumulate;
    uint32_t tiles_n, tiles_m, splits, units, per_xcd, spread;
    float* part;
    unsigned int* counters;
};

template <int T, int NTB, int KG, bool PAIR>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
void linear_tile_kernel(const TileArgs a) {
    constexpr uint32_t RG = 8 / KG, BN = 32 * RG, RT = PAIR ? BN / 2 : BN;
    constexpr uint32_t U = tile_cols(KG), SK = tile_stage(KG), BM = 32 * NTB;
    static_assert(BN == tile_rows(KG) && SK == 64 * KG * U, "tile shape");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    _Float16* const xs = reinterpret_cast<_Float16*>(smem);  // [2][BM][SK], chunks swizzled

    const uint32_t tid = threadIdx.x, lane = tid % 64, n = lane % 32, h = lane / 32;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t rg = wave % RG, kg = wave / RG;

    // Workgroup b runs on XCD b % 8; each XCD takes a contiguous run of (row tile, token tile,
    // split) ids, split fastest.
    const uint32_t L = (blockIdx.x % 8) * a.per_xcd + blockIdx.x / 8;
    if (L >= a.tiles_n * a.tiles_m * a.splits) return;
    const uint32_t split = L % a.splits, tt = (L / a.splits) % a.tiles_m, rt = L / a.splits / a.tiles_m;

    const uint32_t mat = PAIR ? rg / (RG / 2) : rt < a.tile_end[0] ? 0u : rt < a.tile_end[1] ? 1u : 2u;
    const uint8_t* const W = mat == 0 ? a.W[0] : mat == 1 ? a.W[1] : a.W[2];
    float* const out = PAIR || mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : a.out[2];
    const uint32_t n_out = PAIR || mat == 0 ? a.n_out[0] : mat == 1 ? a.n_out[1] : a.n_out[2];
    const uint32_t ld = PAIR || mat == 0 ? a.ld[0] : mat == 1 ? a.ld[1] : a.ld[2];
    const uint32_t rtl = PAIR ? rt : rt - (mat == 0 ? 0u : mat == 1 ? a.tile_end[0] : a.tile_end[1]);
    const uint32_t rowbase = a.row0 + rtl * RT + (PAIR ? rg % (RG / 2) : rg) * 32;  // the wave's rows
    // The token blocks are spread evenly over the token tiles.
    const uint32_t nb = (a.n_tok + 31) / 32;
    const uint32_t tb0 = tile_share0(tt, nb, a.tiles_m), tb1 = tile_share0(tt + 1, nb, a.tiles_m);
    const uint32_t tok0 = 32 * tb0, toks = min(a.n_tok - tok0, 32 * (tb1 - tb0));

    // This split's elements, in units of KG * unit; each k group takes a contiguous share, U steps
    // of 64 elements a stage.
    constexpr uint32_t unit = tile_unit(T);
    const uint32_t u0 = tile_share0(split, a.units, a.splits), units = tile_share0(split + 1, a.units, a.splits) - u0;
    const uint32_t k0 = u0 * KG * unit;
    const uint32_t klen = units * unit, steps = klen / 64, nst = (steps + U - 1) / U;  // per k group
    const bool ragged = k0 + KG * klen > a.n_in || steps % U != 0;  // (elements past the end count as zero)

    // The wave's 32 rows (rows past n_out read the last row and are not written).
    const uint64_t wbase = (uint64_t(min(rowbase, n_out - 1)) * a.row_bytes) & ~uint64_t(15);
    // (the range ends at the 16-byte boundary above the matrix's last byte, in that byte's page)
    const uint64_t left = (uint64_t(n_out) * a.row_bytes - wbase + 15) & ~uint64_t(15);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(W + wbase), 0, int(left < 0x7ffffff0u ? left : 0x7ffffff0u), kBufferFlags);
    using WS = Staged<T, KG>;
    constexpr uint32_t WSB = WS::WK / Fmt<T>::blk * Fmt<T>::bytes, NCH = 32 * WS::CH / 64, QS = WS::WK / 64;
    static_assert(32 * WS::CH % 64 == 0 && WS::CH * 16 <= WS::pitch, "whole rounds of chunks");
    uint8_t* const wsm = smem + tile_x_lds(NTB, KG) + wave * (32 * WS::pitch);
    const uint32_t kg0 = k0 + kg * klen;  // the k group's first element
    auto row_off = [&](uint32_t r) {      // byte of row r's first element of the share
        return uint32_t(uint64_t(min(rowbase + r, n_out - 1)) * a.row_bytes - wbase) + kg0 / Fmt<T>::blk * Fmt<T>::bytes;
    };
    uint32_t wa[NCH], wl[NCH];
    u32x4 wr[NCH];
#pragma unroll
    for (uint32_t i = 0; i < NCH; i++) {
        const uint32_t q = lane + 64 * i, r = q / WS::CH, o = q % WS::CH;
        wa[i] = row_off(r);
        wl[i] = (r * WS::pitch + 16 * o) | o;  // (o < 16: the chunk's place rides along)
    }
    const uint32_t live = min(klen, a.n_in > kg0 ? a.n_in - kg0 : 0u) / 32;  // columns of the share within n_in
    // Where a.spread, the token tiles that share these rows start their walks evenly apart and wrap: each
    // brings a part of the rows into the L2 for all of them (in step they would all wait for HBM at every stage).
    constexpr uint32_t M = QS > U ? QS : U;  // steps of whole W and x stages
    static_assert(M % QS == 0 && M % U == 0, "whole stages");
    uint32_t first = 0;
    if constexpr (KG == 2 && !PAIR)
        if (a.spread && !ragged && steps % M == 0) first = tt * (steps / M) / a.tiles_m * M;
    auto w_stage = [&](uint32_t w) {
        const uint32_t at = w + first / QS;
        return first != 0 && at >= steps / QS ? at - steps / QS : at;
    };
    auto load_w = [&](uint32_t w) {  // W stage w of the walk
        const uint32_t at = w_stage(w) * WSB;
#pragma unroll
        for (uint32_t i = 0; i < NCH; i++) {
            uint32_t off = ((wa[i] + at) & ~15u) + 16 * (wl[i] & 15);
            if constexpr (Fmt<T>::blk == 1)  // (a chunk past the end loads zeros; a block's scale is cleared in col_frag)
                if (w * WS::WK + 16 / Fmt<T>::bytes * (wl[i] & 15) >= 32 * live) off = kOob;
            wr[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, int(off), 0, 0));
        }
    };
    auto store_w = [&]() {
#pragma unroll
        for (uint32_t i = 0; i < NCH; i++) *reinterpret_cast<u32x4*>(wsm + (wl[i] & ~15u)) = wr[i];
    };
    // The raw window of this lane's column of step j (columns 2j + h of the share).
    const uint32_t roff = row_off(n);
    uint32_t wraw[2][Col<T>::ndw], woff[2];
    auto read_w = [&](int s, uint32_t j) {
        const uint32_t i = 2 * (j % QS) + h;
        woff[s] = ((roff + w_stage(j / QS) * WSB) & 15) + col_offset<T>(i);
        col_read<T>(wsm + n * WS::pitch, woff[s], i, wraw[s]);
    };
    auto frag_of = [&](int s, uint32_t j, int e) {
        return col_frag<T>(wraw[s], woff[s], 2 * (j % QS) + h, 2 * j + h < live ? ~0u : 0u, e);
    };

    // x: thread t carries float4 t % FPR of token rows t / FPR + i * RPP (whole lines per row).
    constexpr uint32_t FPR = SK / 4, RPP = 512 / FPR, NX = BM / RPP;
    static_assert(BM % RPP == 0, "x staging");
    typedef _Float16 half4_ __attribute__((ext_vector_type(4)));
    // (16-byte chunks are XOR-swizzled by the row so that 16 rows' reads of one chunk cover the 64
    // banks: a row spans all of them)
    auto xswz = [](uint32_t r) { return r & 15; };
    const uint32_t tr = tid / FPR, tc = tid % FPR;
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.x + size_t(tok0) * a.n_in), 0, int(4 * toks * a.n_in), kBufferFlags);
    const uint32_t xs_ = tc / (16 * U), xi = 4 * (tc % (16 * U));  // k group, element of its slice
    const uint32_t xk = k0 + xs_ * klen + xi;
    float4v xq[NX];
    uint32_t xo[NX];
#pragma unroll
    for (uint32_t i = 0; i < NX; i++) xo[i] = tr + RPP * i < toks ? 4 * ((tr + RPP * i) * a.n_in + xk) : kOob;
    auto load_x = [&](uint32_t j, uint32_t i0, uint32_t i1) {  // pieces i0..i1-1 of stage j
        const uint32_t at = min(j, nst - 1) + first / U;  // (past the walk: its last stage again)
        const uint32_t k = 64 * U * (at >= nst ? at - nst : at);
        const bool cut = ragged && (xi + k >= klen || xk + k >= a.n_in);
#pragma unroll
        for (uint32_t i = 0; i < NX; i++)
            if (i >= i0 && i < i1) xq[i] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
                                                    xrs, int(cut ? kOob : xo[i]), int(4 * k), 0));
    };
    auto store_x = [&](int buf, uint32_t i0, uint32_t i1) {
#pragma unroll
        for (uint32_t i = 0; i < NX; i++) {
            if (i < i0 || i >= i1) continue;
            const uint32_t r = tr + RPP * i;
            half4_ v;
#pragma unroll
            for (int e = 0; e < 4; e++)
                v[e] = _Float16(xq[i][kFragSwap13<T> ? (e == 1 ? 2 : e == 2 ? 1 : e) : e]);
            *reinterpret_cast<half4_*>(xs + buf * (BM * SK) + r * SK + 8 * ((tc / 2) ^ xswz(r)) + 4 * (tc & 1)) = v;
        }
    };

    float16v_ acc[NTB];
#pragma unroll
    for (int b = 0; b < NTB; b++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[b][e] = 0.f;

    // A stage is NG groups of NTB MFMAs. Beside a group's MFMAs the next group's weights are
    // dequantized and its x operands read from LDS, a column's raw bytes are read a column ahead,
    // and the next stage's x goes to the other buffer; the barrier stands before the last group, by
    // when every read of this buffer and every write of the next is done, so that no MFMA waits
    // for an LDS read right behind it. The scheduling barriers keep that order.
    constexpr int NG = 4 * U;
    constexpr uint32_t XPG = (NX + NG - 2) / (NG - 1);  // x pieces per group (none in the last)
    constexpr int kFill = 6;  // VALU instructions between two MFMAs (which issue every 32 cycles)
    half8 wf[2], xa[2][NTB];
    auto read_x = [&](int s, int buf, int i) {
        const uint32_t ch = 8 * (kg * U + i / 4) + 4 * h + i % 4;
#pragma unroll
        for (int b = 0; b < NTB; b++)
            xa[s][b] = *reinterpret_cast<const half8*>(xs + buf * (BM * SK) + (32 * b + n) * SK + 8 * (ch ^ xswz(n)));
    };
    load_x(0, 0, NX);
    load_w(0);
    store_x(0, 0, NX);
    load_x(1, 0, NX);
    store_w();
    load_w(1);
    read_w(0, 0);
    wf[0] = frag_of(0, 0, 0);
    __syncthreads();
    read_x(0, 0, 0);
    for (uint32_t j0 = 0; j0 < nst; j0 += 2) {
#pragma unroll
        for (int jj = 0; jj < 2; jj++) {
            const uint32_t j = j0 + jj;
            if (j >= nst) break;
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const int col = (jj * NG + g) / 4;  // (its parity is the raw window's slot)
                const uint32_t st = j * U + g / 4;
                if (g % 4 == 0) {
                    if ((st + 1) % QS == 0) {  // every column of the W stage has been read
                        store_w();
                        load_w((st + 1) / QS + 1);
                    }
                    read_w((col + 1) & 1, st + 1);
                }
                if (g < NG - 1) read_x((g + 1) & 1, jj, g + 1);
                else read_x(0, jj ^ 1, 0);
                wf[(g + 1) & 1] = frag_of((g % 4 == 3 ? col + 1 : col) & 1, g % 4 == 3 ? st + 1 : st, (g + 1) % 4);
#pragma unroll
                for (int b = 0; b < NTB; b++)
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[g & 1], xa[g & 1][b], acc[b], 0, 0, 0);
                if (g < NG - 1) {
                    store_x(jj ^ 1, g * XPG, g * XPG + XPG);
                    load_x(j + 2, g * XPG, g * XPG + XPG);
                }
                __builtin_amdgcn_sched_group_barrier(0x100, NTB, 0);
#pragma unroll
                for (int b = 0; b < NTB; b++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, kFill, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (g == NG - 2) __syncthreads();
            }
        }
    }
    __syncthreads();

    // Sum the k groups in order: token block b is finished by k group b % KG.
    float* const red = reinterpret_cast<float*>(smem);
    if constexpr (KG > 1) {
        auto slot = [&](uint32_t g, int b) {  // k group g's block b, g != b % KG
            const uint32_t r = g < uint32_t(b % KG) ? g : g - 1;
            return red + (((r * RG + rg) * NTB + b) * 4 * 64 + lane) * 4;
        };
#pragma unroll
        for (int b = 0; b < NTB; b++)
            if (kg != uint32_t(b % KG))
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<float4v*>(slot(kg, b) + q * 256) =
                        float4v{acc[b][4 * q], acc[b][4 * q + 1], acc[b][4 * q + 2], acc[b][4 * q + 3]};
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NTB; b++)
            if (kg == uint32_t(b % KG))
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    float4v s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (uint32_t g = 0; g < KG; g++) {
                        const float4v v = g == uint32_t(b % KG)
                            ? float4v{acc[b][4 * q], acc[b][4 * q + 1], acc[b][4 * q + 2], acc[b][4 * q + 3]}
                            : *reinterpret_cast<const float4v*>(slot(g, b) + q * 256);
                        s = g == 0 ? v : s + v;
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[b][4 * q + e] = s[e];
                }
    }

    if (a.splits > 1) {
        // Publish this split's partial tile with device-scope stores, count its arrival; the last
        // split to arrive sums the partials in split order. Nothing waits for another workgroup.
        const uint32_t tile = rt * a.tiles_m + tt;
        constexpr uint32_t kTileBytes = BN * BM * 4;
        const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
            a.part + size_t(tile) * a.splits * (kTileBytes / 4), 0, int(a.splits * kTileBytes), kBufferFlags);
        auto off = [&](uint32_t sp, int b, int q) {
            return int(sp * kTileBytes + (((rg * NTB + b) * 4 + q) * 64 + lane) * 16);
        };
#pragma unroll
        for (int b = 0; b < NTB; b++)
            if (kg == uint32_t(b % KG))
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4v v = {acc[b][4 * q], acc[b][4 * q + 1], acc[b][4 * q + 2], acc[b][4 * q + 3]};
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), prs, off(split, b, q), 0, kScDevice);
                }
        // The write-through stores are acknowledged before the arrival is counted, and partials
        // are read with device-scope loads; the compiler-only fences keep the order in the code.
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __syncthreads();
        __shared__ unsigned int last;
        if (tid == 0) {
            const unsigned prev = __hip_atomic_fetch_add(a.counters + tile * 16, 1u, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT);
            last = prev == a.splits - 1;
        }
        __syncthreads();
        if (!last) return;
#pragma unroll
        for (int b = 0; b < NTB; b++)
            if (kg == uint32_t(b % KG)) {
                float4v pv[8][4];
#pragma unroll
                for (uint32_t sp = 0; sp < 8; sp++)
                    if (sp < a.splits)
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            pv[sp][q] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(prs, off(sp, b, q), 0, kScDevice));
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    float4v s = pv[0][q];
#pragma unroll
                    for (uint32_t sp = 1; sp < 8; sp++)
                        if (sp < a.splits) s += pv[sp][q];
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[b][4 * q + e] = s[e];
                }
            }
        if (tid == 0)  // leave the workspace ready for the next call
            __hip_atomic_store(a.counters + tile * 16, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    if constexpr (PAIR) {
        // The up waves hand their sums to the gate waves of the same rows and blocks, which form
        // silu(gate) * up as silu_mul_kernel does.
        const uint32_t rp = rg % (RG / 2);
        __syncthreads();  // the reduction's reads are done
#pragma unroll
        for (int b = 0; b < NTB; b++)
            if (kg == uint32_t(b % KG) && mat == 1)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *reinterpret_cast<float4v*>(red + (((rp * NTB + b) * 4 + q) * 64 + lane) * 4) =
                        float4v{acc[b][4 * q], acc[b][4 * q + 1], acc[b][4 * q + 2], acc[b][4 * q + 3]};
        __syncthreads();
        if (mat == 1) return;
#pragma unroll
        for (int b = 0; b < NTB; b++)
            if (kg == uint32_t(b % KG))
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float4v u = *reinterpret_cast<const float4v*>(red + (((rp * NTB + b) * 4 + q) * 64 + lane) * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float g = acc[b][4 * q + e];
                        acc[b][4 * q + e] = g / (1.0f + expf(-g)) * u[e];
                    }
                }
    }

    // A lane holds token n of a block and rows 8q + 4h + 0..3: four consecutive floats of out.
    typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int b = 0; b < NTB; b++) {
        const uint32_t t = 32 * b + n;
        if (kg != uint32_t(b % KG) || t >= toks) continue;
        float* o = out + size_t(tok0 + t) * ld + rowbase + 4 * h;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t r = rowbase + 8 * q + 4 * h;
            const float4v v = {acc[b][4 * q], acc[b][4 * q + 1], acc[b][4 * q + 2], acc[b][4 * q + 3]};
            if (r + 4 <= n_out) {
                float4u* p = reinterpret_cast<float4u*>(o + 8 * q);
                *p = a.accumulate ? *p + v : v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (r + e < n_out) o[8 * q + e] = a.accumulate ? o[8 * q + e] + v[e] : v[e];
            }
        }
    }
}

template <int T, int NTB, int KG, bool PAIR>
int launch(const TileArgs& a, dim3 grid, hipStream_t stream) {
    constexpr size_t lds = tile_lds(NTB, KG, 256 * Staged<T, KG>::pitch);
    static_assert(lds + 16 <= 160 * 1024, "LDS");
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&linear_tile_kernel<T, NTB, KG, PAIR>),
        hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (attr != hipSuccess) return -4;
    hipLaunchKernelGGL((linear_tile_kernel<T, NTB, KG, PAIR>), grid, dim3(512), lds, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

}  // namespace

template <int T>
int launch_tile(const TileCall& c) {
    const uint32_t kg = c.shape.kg, ntb = c.shape.ntb;
    // The kernel's offsets are 32 bits, below kOob: where a tile's tokens or a wave's 32 rows pass
    // that (rows of 67 MB on), a call runs in pieces of fewer of them. The sums keep their order.
    constexpr uint64_t kReach = 0x7ffffff0;
    const uint64_t row_bytes = uint64_t(c.n_in) / Fmt<T>::blk * Fmt<T>::bytes, x_bytes = 4 * uint64_t(c.n_in);
    const uint32_t longest = std::max(c.n_out[0], std::max(c.n_mats > 1 ? c.n_out[1] : 0, c.n_mats > 2 ? c.n_out[2] : 0));
    if (x_bytes > kReach || row_bytes > kReach) return -1;
    if (std::min(c.n_tok, 32 * ntb) * x_bytes > kReach) {
        const uint32_t step = uint32_t(kReach / x_bytes);
        for (uint32_t t = 0; t < c.n_tok; t += step) {
            TileCall p = c;
            p.x += size_t(t) * c.n_in;
            p.n_tok = std::min(step, c.n_tok - t);
            for (uint32_t m = 0; m < c.n_mats; m++) p.out[m] += size_t(t) * c.n_out[m];
            const int rc = launch_tile<T>(p);
            if (rc != 0) return rc;
        }
        return 0;
    }
    if (std::min(std::min(longest, c.rows), 32u) * row_bytes > kReach) {
        const uint32_t step = uint32_t(kReach / row_bytes);
        for (uint32_t r = 0; r < longest; r += step) {
            TileCall p = c;
            p.row0 = r;
            p.rows = step;
            const int rc = launch_tile<T>(p);
            if (rc != 0) return rc;
        }
        return 0;
    }
    TileArgs a{};
    const uint32_t rows = tile_rows(kg) / (c.pair ? 2 : 1);
    a.row0 = c.row0;
    for (uint32_t m = 0; m < 3; m++) {
        a.W[m] = m < c.n_mats ? c.W[m] : nullptr;
        a.out[m] = m < c.n_mats ? c.out[m] : nullptr;
        a.ld[m] = m < c.n_mats ? c.n_out[m] : 0;
        const uint32_t here = a.ld[m] > c.row0 ? std::min(a.ld[m] - c.row0, c.rows) : 0;
        a.n_out[m] = c.row0 + here;
        if (!(c.pair && m > 0)) a.tiles_n += (here + rows - 1) / rows;
        if (m < 2) a.tile_end[m] = a.tiles_n;
    }
    a.x = c.x;
    a.n_in = c.n_in;
    a.n_tok = c.n_tok;
    a.row_bytes = c.n_in / Fmt<T>::blk * Fmt<T>::bytes;
    a.accumulate = c.accumulate;
    a.tiles_m = ((c.n_tok + 31) / 32 + ntb - 1) / ntb;
    a.units = tile_units(T, c.n_in, kg);
    a.splits = c.shape.splits;
    a.spread = c.spread && tile_spread(c.shape, uint64_t(c.n_out[0]) * row_bytes, c.n_tok * x_bytes);
    if (a.splits == 0 || a.splits > std::min(a.units, 8u)) return -1;
    const uint64_t total = uint64_t(a.tiles_n) * a.tiles_m * a.splits, per_xcd = (total + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffu) return -1;
    a.per_xcd = uint32_t(per_xcd);
    a.counters = static_cast<unsigned int*>(c.workspace);
    a.part = a.splits > 1 ? reinterpret_cast<float*>(static_cast<char*>(c.workspace) + kLinearCounterBytes) : nullptr;
    const dim3 grid(uint32_t(per_xcd * 8));
    switch (kg * 8 + ntb) {
// (the shapes without a kernel: tile_cost of linear_shape.h)
#define INGOT_SHAPE(KGv, NTBv)                                         \
    case KGv * 8 + NTBv:                                               \
        if constexpr (T != kF32 || (NTBv < 4 && KGv * NTBv != 12))     \
            return c.pair ? launch<T, NTBv, KGv, true>(a, grid, c.stream) : launch<T, NTBv, KGv, false>(a, grid, c.stream); \
        else return -1
        INGOT_SHAPE(4, 1);
        INGOT_SHAPE(4, 2);
        INGOT_SHAPE(4, 3);
        INGOT_SHAPE(2, 2);
        INGOT_SHAPE(2, 3);
        INGOT_SHAPE(2, 4);
        INGOT_SHAPE(1, 2);
        INGOT_SHAPE(1, 3);
        INGOT_SHAPE(1, 4);
#undef INGOT_SHAPE
        default: return -1;
    }
}

template int launch_tile<INGOT_TILE_TYPE>(const TileCall& c);

}  // namespace ingot
