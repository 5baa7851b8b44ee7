// linear_formats.h — the GGUF weight formats as the gfx950 linear kernels read them: block sizes,
// and the loads of one 32-element column of a row from its dword-aligned window.
#pragma once

#include "attn_common.h"
#include "attn_internal.h"

namespace ingot {

namespace {

typedef float float16v_ __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kBufferFlags = 0x00020000;  // buffer descriptor word 3 (raw, 32-bit format)

// ---------------------------------------------------------------- block formats

// GGUF type ids (ggml's enum, src/gguf.h:30-33).
enum : int { kF32 = 0, kF16 = 1, kQ4_0 = 2, kQ4_1 = 3, kQ8_0 = 8, kQ6_K = 14, kBF16 = 30 };

__device__ __forceinline__ float f16_bits(uint32_t h) {
    return float(__builtin_bit_cast(_Float16, uint16_t(h)));
}
__device__ __forceinline__ uint32_t ld_u16(const uint8_t* p) {
    return *reinterpret_cast<const uint16_t*>(p);
}
// 8 bytes from a 2-byte aligned address.
__device__ __forceinline__ void ld_8bytes(const uint8_t* p, uint32_t& lo, uint32_t& hi) {
    lo = ld_u16(p) | (ld_u16(p + 2) << 16);
    hi = ld_u16(p + 4) | (ld_u16(p + 6) << 16);
}
__device__ __forceinline__ uint32_t byte_of(uint32_t lo, uint32_t hi, int i) {
    return ((i < 4 ? lo : hi) >> (8 * (i & 3))) & 0xFF;
}

template <int T> struct Fmt;
template <> struct Fmt<kF32>  { static constexpr uint32_t blk = 1,   bytes = 4; };
template <> struct Fmt<kF16>  { static constexpr uint32_t blk = 1,   bytes = 2; };
template <> struct Fmt<kBF16> { static constexpr uint32_t blk = 1,   bytes = 2; };
template <> struct Fmt<kQ8_0> { static constexpr uint32_t blk = 32,  bytes = 34; };
template <> struct Fmt<kQ4_0> { static constexpr uint32_t blk = 32,  bytes = 18; };
template <> struct Fmt<kQ4_1> { static constexpr uint32_t blk = 32,  bytes = 20; };
template <> struct Fmt<kQ6_K> { static constexpr uint32_t blk = 256, bytes = 210; };

// A lane's column (32 consecutive elements of a row) is loaded as the dword-aligned window around
// it: a quantized block is only 2-byte aligned.
template <int T> struct Col;
template <> struct Col<kQ4_0> { static constexpr int ndw = 5, bytes = 18; };
template <> struct Col<kQ4_1> { static constexpr int ndw = 5, bytes = 20; };
template <> struct Col<kQ8_0> { static constexpr int ndw = 9, bytes = 34; };
template <> struct Col<kF16>  { static constexpr int ndw = 16, bytes = 64; };
template <> struct Col<kBF16> { static constexpr int ndw = 16, bytes = 64; };
template <> struct Col<kF32>  { static constexpr int ndw = 32, bytes = 128; };
// Q6_K: column c is the 32-element group (h, g) = ((c % 8) / 4, c % 4) of 210-byte block c / 8;
// the lane loads the windows of its 32 low-bit bytes, its 32 high-bit bytes, its two scales and
// the block's d.
template <> struct Col<kQ6_K> { static constexpr int ndw = 20; };

template <int T>
constexpr bool kStreamed = T == kQ4_0 || T == kQ4_1 || T == kQ8_0 || T == kF16 || T == kBF16 || T == kQ6_K;

// Byte offset of column c from the row start.
template <int T>
__device__ __forceinline__ uint32_t col_offset(uint32_t c) {
    if constexpr (T == kQ6_K) return 210 * (c >> 3);
    else return c * Col<T>::bytes;
}

// The window of the column at byte offset off (relative to a 16-byte aligned buffer base).
template <int T>
__device__ __forceinline__ void col_load(const __amdgpu_buffer_rsrc_t& rs, uint32_t off, uint32_t (&w)[Col<T>::ndw],
                                         uint32_t c = 0) {
    auto ld4 = [&](uint32_t o, int at) {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, int(o), 0, 0));
        w[at] = v[0]; w[at + 1] = v[1]; w[at + 2] = v[2]; w[at + 3] = v[3];
    };
    if constexpr (T == kQ6_K) {
        const uint32_t h = (c >> 2) & 1, g = c & 3;
        const uint32_t pl = (off + 64 * h + 32 * (g & 1)) & ~3u, ph = (off + 128 + 32 * h) & ~3u;
        ld4(pl, 0);
        ld4(pl + 16, 4);
        w[8] = __builtin_amdgcn_raw_buffer_load_b32(rs, int(pl + 32), 0, 0);
        ld4(ph, 9);
        ld4(ph + 16, 13);
        w[17] = __builtin_amdgcn_raw_buffer_load_b32(rs, int(ph + 32), 0, 0);
        w[18] = __builtin_amdgcn_raw_buffer_load_b32(rs, int((off + 192 + 8 * h + 2 * g) & ~3u), 0, 0);
        w[19] = __builtin_amdgcn_raw_buffer_load_b32(rs, int((off + 208) & ~3u), 0, 0);
    } else if constexpr (T == kF16 || T == kBF16) {
        for (int i = 0; i < 4; i++) ld4(off + 16 * i, 4 * i);
    } else {
        const uint32_t p = off & ~3u;
        ld4(p, 0);
        if constexpr (T == kQ8_0) ld4(p + 16, 4);
        w[Col<T>::ndw - 1] = __builtin_amdgcn_raw_buffer_load_b32(rs, int(p + 4 * (Col<T>::ndw - 1)), 0, 0);
    }
}

// Block types whose B fragments hold their 8 k values in the order 0,2,1,3,4,6,5,7: two
// elements two bytes apart share a 32-bit word, so one masked word gives a packed half pair.
template <int T>
constexpr bool kFragSwap13 = T == kQ4_0 || T == kQ8_0;

__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t c) {
    return (a & m) | c;  // v_and_or_b32
}

}  // namespace

}  // namespace ingot
