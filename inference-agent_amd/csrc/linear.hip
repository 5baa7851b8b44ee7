// linear.hip — out (+)= W·x over GGUF weight layouts, for gfx950.
//
// The projection right after attention (wo with the residual accumulate, src/metal_backend.mm:
// 446-447; src/cpu_backend.cpp:71-72) and every other linear layer of the forward pass
// (src/metal_backend.mm:282-310). W keeps its on-disk layout: ne = [n_in, n_out], row r holds
// n_in elements in blocks of the tensor type (src/ops.cpp:33-87 for the block formats).
// x is f32 [n_tok][n_in]; out is f32 [n_tok][n_out] starting at out + out_offset.
//
// One token (decode): linear_matvec_kernel. The op is HBM-bound (each weight byte used once).
// A workgroup copies the contiguous bytes of its rows into LDS with 16-byte loads (quantized
// blocks are only 2-byte aligned, so parsing them straight from HBM would need 2-byte loads),
// then every wave takes a quarter of the row length for all of the rows, with its slice of x in
// registers, and dequantizes 8 elements at a time from LDS in f32. Arithmetic is f32 throughout,
// like the CPU path (src/ops.cpp:199-224) and the Metal matvec kernels (shaders/kernels.metal:
// 73-226).
//
// Several tokens (prefill): linear_tile.hip, whose workgroup shape is chosen here.
#include <algorithm>
#include <type_traits>

#include "linear_formats.h"
#include "linear_shape.h"

namespace ingot {

namespace {

// Elements k..k+7 (k % 8 == 0) of the row starting at `row`, dequantized to f32.
// Q8_0 (34 B / 32): d·q.  Q4_0 (18 B / 32): byte j holds element j (low nibble) and j+16
// (high nibble), d·(nibble-8).  Q4_1 (20 B / 32): d·nibble + m.  Q6_K (210 B / 256): ql[128]
// low 4 bits, qh[64] high 2 bits, 16 int8 scales, f16 d; within each 128-element half, element
// 32g + l (g = 0..3, l = 0..31) takes the low (g < 2) or high nibble of ql[l + 32(g&1)] and
// bits 2g..2g+1 of qh[l], with scale index l/16 + 2g: d·scale·(q6-32).
template <int T>
__device__ __forceinline__ void deq8(const uint8_t* row, uint32_t k, float w[8]) {
    if constexpr (T == kF32) {
        const float4v a = *reinterpret_cast<const float4v*>(row + 4 * k);
        const float4v b = *reinterpret_cast<const float4v*>(row + 4 * k + 16);
        for (int i = 0; i < 4; i++) { w[i] = a[i]; w[i + 4] = b[i]; }
    } else if constexpr (T == kF16) {
        const half8 h = *reinterpret_cast<const half8*>(row + 2 * k);
        for (int i = 0; i < 8; i++) w[i] = float(h[i]);
    } else if constexpr (T == kBF16) {
        const u32x4 u = *reinterpret_cast<const u32x4*>(row + 2 * k);
        for (int i = 0; i < 4; i++) {
            w[2 * i] = __uint_as_float(u[i] << 16);
            w[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u);
        }
    } else if constexpr (T == kQ8_0) {
        const uint8_t* b = row + 34 * (k / 32);
        const float d = f16_bits(ld_u16(b));
        uint32_t lo, hi;
        ld_8bytes(b + 2 + k % 32, lo, hi);
        for (int i = 0; i < 8; i++) w[i] = d * float(int8_t(byte_of(lo, hi, i)));
    } else if constexpr (T == kQ4_0 || T == kQ4_1) {
        constexpr int kBytes = T == kQ4_0 ? 18 : 20, kQs = T == kQ4_0 ? 2 : 4;
        const uint8_t* b = row + kBytes * (k / 32);
        const uint32_t off = k % 32;
        const float d = f16_bits(ld_u16(b));
        const float m = T == kQ4_1 ? f16_bits(ld_u16(b + 2)) : -8.f * d;
        uint32_t lo, hi;
        ld_8bytes(b + kQs + (off & 15), lo, hi);
        const int sh = off >= 16 ? 4 : 0;
        for (int i = 0; i < 8; i++) w[i] = d * float((byte_of(lo, hi, i) >> sh) & 0xF) + m;
    } else if constexpr (T == kQ6_K) {
        const uint8_t* b = row + 210 * (k / 256);
        const uint32_t e = k % 256, h = e / 128, g = (e % 128) / 32, l = e % 32;
        const float d = f16_bits(ld_u16(b + 208));
        const float s = d * float(int8_t(b[192 + h * 8 + l / 16 + 2 * g]));
        uint32_t ql0, ql1, qh0, qh1;
        ld_8bytes(b + h * 64 + 32 * (g & 1) + l, ql0, ql1);
        ld_8bytes(b + 128 + h * 32 + l, qh0, qh1);
        const int shl = g >= 2 ? 4 : 0, shh = 2 * int(g);
        for (int i = 0; i < 8; i++) {
            const int q = int(((byte_of(ql0, ql1, i) >> shl) & 0xF) |
                              (((byte_of(qh0, qh1, i) >> shh) & 3) << 4));
            w[i] = s * float(q - 32);
        }
    }
}

// dot(elements k..k+7 of the row, x0|x1) for the block types, without materializing each
// weight: the group's quants are converted a byte at a time (unsigned bytes, so Q8_0's int8 are
// biased by +128) and the block offset/scale applied once per group:
//   Q4_0  d * (sum q x - 8 sum x)      Q4_1  d * sum q x + m * sum x
//   Q8_0  d * (sum (q+128) x - 128 sum x)
// The same value as the per-element form up to f32 rounding (CPU dot_q4_0 / dot_q8_0 also sum
// the integer products per block and scale once, src/ops.cpp:153-187).
template <int T>
__device__ __forceinline__ float bytes_dot4(uint32_t w, const float4v& x) {
    float s = float(w & 0xFF) * x[0];
    s += float((w >> 8) & 0xFF) * x[1];
    s += float((w >> 16) & 0xFF) * x[2];
    s += float(w >> 24) * x[3];
    return s;
}

template <int T>
__device__ __forceinline__ float dot8(const uint8_t* row, uint32_t k, const float4v& x0, const float4v& x1) {
    const float sx = ((x0[0] + x0[1]) + (x0[2] + x0[3])) + ((x1[0] + x1[1]) + (x1[2] + x1[3]));
    if constexpr (T == kQ8_0) {
        const uint8_t* b = row + 34 * (k / 32);
        const float d = f16_bits(ld_u16(b));
        uint32_t lo, hi;
        ld_8bytes(b + 2 + k % 32, lo, hi);
        const float s = bytes_dot4<T>(lo ^ 0x80808080u, x0) + bytes_dot4<T>(hi ^ 0x80808080u, x1);
        return d * (s - 128.f * sx);
    } else {
        constexpr int kBytes = T == kQ4_0 ? 18 : 20, kQs = T == kQ4_0 ? 2 : 4;
        const uint8_t* b = row + kBytes * (k / 32);
        const uint32_t off = k % 32;
        const float d = f16_bits(ld_u16(b));
        uint32_t lo, hi;
        ld_8bytes(b + kQs + (off & 15), lo, hi);
        const uint32_t sh = off >= 16 ? 4 : 0;
        const float s = bytes_dot4<T>((lo >> sh) & 0x0F0F0F0Fu, x0) + bytes_dot4<T>((hi >> sh) & 0x0F0F0F0Fu, x1);
        if constexpr (T == kQ4_0) return d * (s - 8.f * sx);
        else return d * s + f16_bits(ld_u16(b + 2)) * sx;
    }
}

__device__ __forceinline__ float wave_sum(float x) {
    x = row16_sum(x);
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
    return x;
}

// ---------------------------------------------------------------- one token

constexpr uint32_t kMvLdsBytes = 160 * 1024;  // weight rows + x staged per workgroup (at most)
constexpr int kMvChunks = 8;  // 16-byte staging loads per thread per round (one round up to 32 KB)

// What happens to x before the products, and to the row sums after (ingot_proj):
//   prologue kProNone: x as given; kProRmsNorm: x * (1/sqrt(mean(x^2) + eps)) * aux, the
//     rmsnorm that precedes q/k/v and gate/up (the same arithmetic, in the same order, as
//     rmsnorm_kernel, so the fused and the separate sequence give identical results);
//   epilogue kEpiStore / kEpiAccumulate: out = s or out += s per matrix; kEpiSiluGate: two
//     matrices (gate, up) over the same rows, out0 = silu(s_gate) * s_up with
//     silu(g) = g / (1 + exp(-g)), as silu_mul_kernel.
enum : int { kProNone = 0, kProRmsNorm = 1 };
enum : int { kEpiStore = 0, kEpiAccumulate = 1, kEpiSiluGate = 2, kEpiRopeKv = 3 };
//   kEpiRopeKv: matrices q, k, v of one decode token: q and k rotated by RoPE (pairs (2i, 2i+1)
//     of each head, angle pos * inv_freq[i], rotated as rope_kv_store_kernel does), q stored in
//     f32, K and V rounded to f16 into their cache rows (ingot_rope_kv_store's work).

// Up to three matrices of one type sharing n_in and x (q/k/v, gate/up), launched as one grid:
// blocks [blk_end[m-1], blk_end[m]) take matrix m's rows, R per block.
struct MvArgs {
    const uint8_t* W[3];
    float* out[3];
    uint32_t n_out[3];
    uint32_t blk_end[3];
    const float* x;
    const float* aux;  // rmsnorm weights [n_in]
    uint32_t n_in, row_bytes;
    uint32_t blocks;  // linear_stream_kernel: row blocks of the call (the grid may be smaller)
    float eps;
    // kEpiRopeKv
    const float* inv_freq;
    _Float16* cache[2];  // K and V rows of the token
    uint32_t head_dim, pos;
};

// R weight rows per matrix per workgroup of 4 waves (2R for the gate/up pair); each wave takes a
// quarter of the 8-element groups of all rows, reads x for a group once and applies it to every
// row (x dominates the LDS reads otherwise: 32 bytes per group against ~10 for a Q4_0 row). x
// (and the rmsnorm weights), and for the block-quantized types the rows' bytes, are staged in
// LDS by one pass of 16-byte loads, all issued before the first wait; rows of plain
// F32/F16/BF16 elements (every group a 16- or 32-byte aligned piece) are read straight from
// memory. Rows past n_out are computed from a clamped row and not written.
template <int T>
constexpr bool kMvStageW = !(T == kF32 || T == kF16 || T == kBF16);

template <int T, int R, int PRO, int EPI>
__global__ __launch_bounds__(256) void linear_matvec_kernel(const MvArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int NS = EPI == kEpiSiluGate ? 2 : 1;  // row sets: (gate, up) or one matrix
    constexpr int NR = NS * R;
    const uint32_t tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    uint32_t m = 0, blk = blockIdx.x;
    if constexpr (EPI != kEpiSiluGate) {
        if (blk >= a.blk_end[0]) m = blk >= a.blk_end[1] ? 2 : 1;
        if (m > 0) blk -= a.blk_end[m - 1];
    }
    const uint32_t n_in = a.n_in, row_bytes = a.row_bytes;
    const uint32_t n_out = a.n_out[m];
    const uint32_t row0 = blk * R;
    const uint32_t nrows = min(uint32_t(R), n_out - row0);

    // LDS: x ([n_in] f32, 16-byte chunks), the rmsnorm weights, then each set's rows' bytes
    // from a 16-byte aligned start.
    const uint32_t xchunks = n_in / 4;
    const uint32_t achunks = PRO == kProRmsNorm ? xchunks : 0;
    const uint64_t start = uint64_t(row0) * row_bytes;
    const uint64_t a0 = start & ~uint64_t(15);
    const uint32_t shift = uint32_t(start - a0);
    const uint32_t wchunks = kMvStageW<T> ? (shift + nrows * row_bytes + 15) / 16 : 0;
    const uint32_t nchunks = xchunks + achunks + NS * wchunks;
    const uint64_t w_bytes = uint64_t(n_out) * row_bytes;
    // Bytes from a0 to the end of the matrix, rounded up to whole dwords: buffer loads drop
    // every dword that reaches past num_records, and a row may end mid-dword (an odd number of
    // 18-, 34- or 210-byte rows); the dword holding the last byte never crosses a page.
    const uint64_t left = (w_bytes - a0 + 3) & ~uint64_t(3);
    const int wrec = int(left < 0x7fffffffu ? left : 0x7fffffffu);
    __amdgpu_buffer_rsrc_t ws[NS];
#pragma unroll
    for (int s = 0; s < NS; s++)
        ws[s] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.W[m + s] + a0), 0, wrec, kBufferFlags);
    const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x), 0,
                                                                        int(4 * n_in), kBufferFlags);
    const __amdgpu_buffer_rsrc_t as = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(PRO == kProRmsNorm ? a.aux : a.x), 0, int(4 * n_in), kBufferFlags);
    // The staging rounds walk the regions x | norm weights | row set 0 | row set 1, each padded
    // to a multiple of 256 chunks, so that a load's source (its buffer descriptor) is uniform
    // across the workgroup: a descriptor chosen per lane makes the compiler loop over the
    // distinct descriptors of a wave.
    const uint32_t px = (xchunks + 255) & ~255u, pa = (achunks + 255) & ~255u, pw = (wchunks + 255) & ~255u;
    const uint32_t nvirt = px + pa + NS * pw;
    for (uint32_t base = 0; base < nvirt; base += 256 * kMvChunks) {
        u32x4 st[kMvChunks];
        uint32_t dst[kMvChunks];
#pragma unroll
        for (int i = 0; i < kMvChunks; i++) {
            const uint32_t v0 = base + 256u * i;  // workgroup-uniform
            if (v0 >= nvirt) break;
            // region of this round slot, its chunk count, LDS chunk offset and descriptor
            uint32_t start, count, lds0;
            __amdgpu_buffer_rsrc_t src;
            if (v0 < px) {
                start = 0; count = xchunks; lds0 = 0; src = xs;
            } else if (v0 < px + pa) {
                start = px; count = achunks; lds0 = xchunks; src = as;
            } else if (NS == 1 || v0 < px + pa + pw) {
                start = px + pa; count = wchunks; lds0 = xchunks + achunks; src = ws[0];
            } else {
                start = px + pa + pw; count = wchunks; lds0 = xchunks + achunks + wchunks; src = ws[NS - 1];
            }
            const uint32_t local = v0 - start + tid;
            st[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, int(16 * min(local, count - 1)), 0, 0));
            dst[i] = local < count ? lds0 + local : ~0u;
        }
#pragma unroll
        for (int i = 0; i < kMvChunks; i++) {
            if (base + 256u * i >= nvirt) break;
            if (dst[i] != ~0u) *reinterpret_cast<u32x4*>(smem + 16 * dst[i]) = st[i];
        }
    }
    float* red = reinterpret_cast<float*>(smem + 16 * nchunks);  // [4 waves][NR]
    __syncthreads();

    float* xl = reinterpret_cast<float*>(smem);
    if constexpr (PRO == kProRmsNorm) {
        // rmsnorm_kernel's reduction: float4 per thread strided by 1024 elements, row sums,
        // then the four wave partials in fixed order; each thread then rescales the elements
        // it summed.
        const float* wl = xl + n_in;
        float ss = 0.f;
        for (uint32_t i = 4 * tid; i < n_in; i += 1024) {
            const float4v v = *reinterpret_cast<const float4v*>(xl + i);
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        ss = row16_sum(ss);
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        const float total = (red[0] + red[1]) + (red[2] + red[3]);
        const float scale = 1.0f / sqrtf(total / float(n_in) + a.eps);
        for (uint32_t i = 4 * tid; i < n_in; i += 1024) {
            const float4v v = *reinterpret_cast<const float4v*>(xl + i);
            const float4v g = *reinterpret_cast<const float4v*>(wl + i);
            *reinterpret_cast<float4v*>(xl + i) = v * scale * g;
        }
        __syncthreads();
    }

    const uint32_t groups = n_in / 8, per_wave = (groups + 3) / 4;
    const uint32_t g_begin = wave * per_wave, g_end = min(groups, g_begin + per_wave);
    float acc[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) acc[r] = 0.f;
    if constexpr (kMvStageW<T>) {
        const uint8_t* rows = smem + 16 * (xchunks + achunks) + shift;
        for (uint32_t g = g_begin + lane; g < g_end; g += 64) {
            const float4v x0 = *reinterpret_cast<const float4v*>(xl + 8 * g);
            const float4v x1 = *reinterpret_cast<const float4v*>(xl + 8 * g + 4);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                const uint8_t* row = rows + (r / R) * 16 * wchunks + min(uint32_t(r % R), nrows - 1) * row_bytes;
                if constexpr (T == kQ8_0 || T == kQ4_0 || T == kQ4_1) {
                    acc[r] += dot8<T>(row, 8 * g, x0, x1);
                } else {
                    float w[8];
                    deq8<T>(row, 8 * g, w);
                    float s = 0.f;
                    for (int i = 0; i < 4; i++) s += w[i] * x0[i];
                    for (int i = 0; i < 4; i++) s += w[i + 4] * x1[i];
                    acc[r] += s;
                }
            }
        }
    } else {
        constexpr uint32_t GB = T == kF32 ? 32 : 16;  // bytes per 8-element group
        __amdgpu_buffer_rsrc_t rs[NS];
#pragma unroll
        for (int s = 0; s < NS; s++)
            rs[s] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.W[m + s] + start), 0,
                                                      int(nrows * row_bytes), kBufferFlags);
        for (uint32_t g = g_begin + lane; g < g_end; g += 64) {
            u32x4 raw[NR][GB / 16];
#pragma unroll
            for (int r = 0; r < NR; r++)
                for (uint32_t q = 0; q < GB / 16; q++)
                    raw[r][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                             rs[r / R], int(min(uint32_t(r % R), nrows - 1) * row_bytes + g * GB + 16 * q), 0, 0));
            const float4v x0 = *reinterpret_cast<const float4v*>(xl + 8 * g);
            const float4v x1 = *reinterpret_cast<const float4v*>(xl + 8 * g + 4);
#pragma unroll
            for (int r = 0; r < NR; r++) {
                float w[8];
                deq8<T>(reinterpret_cast<const uint8_t*>(&raw[r][0]), 0, w);
                float s = 0.f;
                for (int i = 0; i < 4; i++) s += w[i] * x0[i];
                for (int i = 0; i < 4; i++) s += w[i + 4] * x1[i];
                acc[r] += s;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const float s = wave_sum(acc[r]);
        if (lane == 0) red[wave * NR + r] = s;
    }
    __syncthreads();
    if (tid < nrows) {
        auto total = [&](int r) { return (red[r] + red[NR + r]) + (red[2 * NR + r] + red[3 * NR + r]); };
        float* o = a.out[m] + row0 + tid;
        if constexpr (EPI == kEpiSiluGate) {
            const float g = total(tid), u = total(R + tid);
            *o = g / (1.0f + expf(-g)) * u;
        } else {
            const float s = total(tid);
            *o = EPI == kEpiAccumulate ? *o + s : s;
        }
    }
}

// ---------------------------------------------------------------- one token, streamed rows

// The block types with 32-element blocks and the 16-bit float types take a second one-token
// kernel that reads weight rows straight from memory into registers (no LDS staging, no
// barrier between the loads and the arithmetic): x (after the rmsnorm prologue) is staged in
// LDS once per workgroup; a half-wave (32 lanes) owns RPH rows and walks their 32-element
// columns, lane l taking columns l, l+32, ..., with the next column's loads issued before the
// current column's arithmetic. A quantized block is only 2-byte aligned, so a lane loads the
// dword-aligned window around it (5 dwords for Q4_0 / Q4_1, 9 for Q8_0) and realigns it with
// v_alignbyte. Each x column is read from LDS once per lane and applied to all RPH rows.
// s + sum_k byte_k(q) * x[k], one fma per element (v_cvt_f32_ubyte0..3 read the bytes in place).
__device__ __forceinline__ float fma_u8x4(uint32_t q, const float4v& x, float s) {
    s = fmaf(float(q & 0xFF), x[0], s);
    s = fmaf(float((q >> 8) & 0xFF), x[1], s);
    s = fmaf(float((q >> 16) & 0xFF), x[2], s);
    return fmaf(float(q >> 24), x[3], s);
}

// The low / high nibbles of each byte of w, as bytes. The mask is applied in inline asm so the
// optimizer cannot fold it into the byte extraction of fma_u8x4 (it would turn each
// v_cvt_f32_ubyteN into a bit-field extract plus a conversion).
__device__ __forceinline__ uint32_t lo_nibbles(uint32_t w) {
    uint32_t r;
    asm("v_and_b32 %0, 0x0f0f0f0f, %1" : "=v"(r) : "v"(w));
    return r;
}
__device__ __forceinline__ uint32_t hi_nibbles(uint32_t w) {
    uint32_t r;
    asm("v_lshrrev_b32 %0, 4, %1\n\tv_and_b32 %0, 0x0f0f0f0f, %0" : "=&v"(r) : "v"(w));
    return r;
}

// W-row column · x column (32 elements; sx = sum of the x column, shared by the rows).
template <int T>
__device__ __forceinline__ float col_dot(const uint32_t (&w)[Col<T>::ndw], uint32_t off, const float4v (&x)[8], float sx,
                                         uint32_t c = 0, float sx_hi = 0.f) {
    if constexpr (T == kQ6_K) {
        // q = (4 low bits from ql: the low nibble for g < 2, else the high one) | (2 bits of qh
        // at 2g) << 4, an unsigned 0..63 byte; each 16 elements share an int8 scale:
        // d * (sc_lo * (sum_lo q x - 32 sum_lo x) + sc_hi * (sum_hi q x - 32 sum_hi x)).
        const uint32_t h = (c >> 2) & 1, g = c & 3;
        const uint32_t shl_ = (off + 64 * h + 32 * (g & 1)) & 3, shh_ = (off + 128 + 32 * h) & 3;
        const uint32_t nib = g >= 2 ? 4 : 0, hb = 2 * g;
        float s_lo = 0.f, s_hi = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t ql = __builtin_amdgcn_alignbyte(w[i + 1], w[i], shl_);
            const uint32_t qh = __builtin_amdgcn_alignbyte(w[9 + i + 1], w[9 + i], shh_);
            uint32_t q = ((ql >> nib) & 0x0F0F0F0Fu) | (((qh >> hb) & 0x03030303u) << 4);
            asm("" : "+v"(q));  // keep the byte conversions as v_cvt_f32_ubyteN
            if (i < 4) s_lo = fma_u8x4(q, x[i], s_lo);
            else s_hi = fma_u8x4(q, x[i], s_hi);
        }
        const uint32_t scw = w[18] >> (8 * ((off + 192 + 8 * h + 2 * g) & 3));
        const float sc_lo = float(int8_t(scw & 0xFF)), sc_hi = float(int8_t((scw >> 8) & 0xFF));
        const float d = f16_bits((w[19] >> (8 * ((off + 208) & 3))) & 0xFFFF);
        const float t = fmaf(sc_lo, fmaf(-32.f, sx, s_lo), __fmul_rn(sc_hi, fmaf(-32.f, sx_hi, s_hi)));
        return __fmul_rn(d, t);
    } else if constexpr (T == kF16 || T == kBF16) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const uint32_t u = w[2 * i + e];
                float lo, hi;
                if constexpr (T == kF16) {
                    lo = f16_bits(u & 0xFFFF);
                    hi = f16_bits(u >> 16);
                } else {
                    lo = __uint_as_float(u << 16);
                    hi = __uint_as_float(u & 0xFFFF0000u);
                }
                s = fmaf(lo, x[i][2 * e], s);
                s = fmaf(hi, x[i][2 * e + 1], s);
            }
        }
        return s;
    } else if constexpr (T == kQ4_1) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s = fma_u8x4(lo_nibbles(w[1 + i]), x[i], s);
            s = fma_u8x4(hi_nibbles(w[1 + i]), x[4 + i], s);
        }
        return fmaf(f16_bits(w[0] & 0xFFFF), s, __fmul_rn(f16_bits(w[0] >> 16), sx));
    } else {
        // the block starts at byte 0 or 2 of the window; its quants at byte 2 or 4
        const bool odd = (off & 2) != 0;
        const float d = f16_bits((odd ? w[0] >> 16 : w[0]) & 0xFFFF);
        constexpr int NQ = T == kQ8_0 ? 8 : 4;
        uint32_t q[NQ];
#pragma unroll
        for (int i = 0; i < NQ; i++) q[i] = odd ? w[i + 1] : __builtin_amdgcn_alignbyte(w[i + 1], w[i], 2);
        float s = 0.f;
        if constexpr (T == kQ8_0) {
#pragma unroll
            for (int i = 0; i < 8; i++) s = fma_u8x4(q[i] ^ 0x80808080u, x[i], s);
            return __fmul_rn(d, fmaf(-128.f, sx, s));
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s = fma_u8x4(lo_nibbles(q[i]), x[i], s);
                s = fma_u8x4(hi_nibbles(q[i]), x[4 + i], s);
            }
            return __fmul_rn(d, fmaf(-8.f, sx, s));
        }
    }
}

// x chunk (16 bytes) i of the staged x -> its LDS slot: column c = i / 8 keeps its 8 chunks,
// permuted by (c / 2) % 8, so that the 16 lanes of one LDS read phase (consecutive columns,
// same chunk) hit 16 different 16-byte bank groups.
__device__ __forceinline__ uint32_t xslot(uint32_t i) {
    const uint32_t c = i >> 3;
    return (c << 3) | ((i & 7) ^ ((c >> 1) & 7));
}

template <int T, int RPH, int PRO, int EPI, int NT, bool LOOP>
__global__ __launch_bounds__(NT) void linear_stream_kernel(const MvArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int NDW = Col<T>::ndw;
    constexpr int RPM = EPI == kEpiSiluGate ? RPH / 2 : RPH;  // rows of each matrix per half-wave
    const uint32_t tid = threadIdx.x, lane = tid % 64, hw = tid / 32, l32 = tid % 32;
    const uint32_t n_in = a.n_in, row_bytes = a.row_bytes;
    constexpr uint32_t NHW = NT / 32;  // half-waves

    // The rows of block blk of the call: this half-wave's RPM rows of matrix m from row0 on (and
    // the same RPM of matrix m + 1 for the gate/up pair); rows past n_out read the last row and are
    // not written. With LOOP (many more blocks than the chip holds workgroups) a workgroup takes
    // blocks blockIdx.x, blockIdx.x + gridDim.x, ... and stages x once for all of them.
    uint32_t blk = blockIdx.x, m, n_out, row0;
    uint32_t roff[RPH];
    __amdgpu_buffer_rsrc_t rs[EPI == kEpiSiluGate ? 2 : 1];
    auto take_block = [&]() {
        uint32_t local = blk;
        m = 0;
        if constexpr (EPI != kEpiSiluGate) {
            if (local >= a.blk_end[0]) m = local >= a.blk_end[1] ? 2 : 1;
            if (m > 0) local -= a.blk_end[m - 1];
        }
        n_out = a.n_out[m];
        row0 = local * NHW * RPM;
        const uint64_t wbase = (uint64_t(row0) * row_bytes) & ~uint64_t(15);
#pragma unroll
        for (int i = 0; i < RPH; i++) {
            const uint32_t r = min(row0 + hw * RPM + uint32_t(i % RPM), n_out - 1);
            roff[i] = uint32_t(uint64_t(r) * row_bytes - wbase);
        }
        const uint64_t left = (uint64_t(n_out) * row_bytes - wbase + 3) & ~uint64_t(3);
        const int nrec = int(left < 0x7fffffffu ? left : 0x7fffffffu);
        rs[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.W[m] + wbase), 0, nrec, kBufferFlags);
        if constexpr (EPI == kEpiSiluGate)
            rs[1] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.W[1] + wbase), 0, nrec, kBufferFlags);
    };
    take_block();

    const uint32_t ncols = n_in / 32, last = ncols - 1;
    const uint32_t nsteps = (ncols + 31) / 32;
    uint32_t b0[RPH][NDW], b1[RPH][NDW], b2[RPH][NDW];
    auto load = [&](uint32_t step, uint32_t (&b)[RPH][NDW]) {
        const uint32_t c = min(step * 32 + l32, last);
#pragma unroll
        for (int i = 0; i < RPH; i++) col_load<T>(rs[i / RPM], roff[i] + col_offset<T>(c), b[i], c);
    };
    // x (and the norm weights, unpermuted after it) into LDS. The loads of x's first round go
    // out first, then the first three columns of the rows (they do not depend on x), then x is
    // stored: the row data streams in while x is staged and normalized.
    const uint32_t xchunks = n_in / 4;
    const uint32_t nchunks = PRO == kProRmsNorm ? 2 * xchunks : xchunks;
    float4v* xl = reinterpret_cast<float4v*>(smem);
    const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x), 0,
                                                                        int(4 * n_in), kBufferFlags);
    const __amdgpu_buffer_rsrc_t as = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(PRO == kProRmsNorm ? a.aux : a.x), 0, int(4 * n_in), kBufferFlags);
    auto stage_round = [&](uint32_t base, bool prefetch) {
        float4v st[kMvChunks];
        // (x chunks and norm-weight chunks come from two descriptors; the choice is made per
        // load from the workgroup-uniform round position, never per lane, which would make the
        // compiler loop over the distinct descriptors of a wave)
#pragma unroll
        for (int i = 0; i < kMvChunks; i++) {
            if (base + NT * i >= nchunks) break;  // workgroup-uniform
            const uint32_t c = min(base + tid + NT * i, nchunks - 1);
            const uint32_t cx = min(c, xchunks - 1);
            const float4v vx = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(xs, int(16 * cx), 0, 0));
            if (PRO == kProRmsNorm && base + NT * i + NT - 1 >= xchunks) {
                const uint32_t ca = c >= xchunks ? c - xchunks : 0;
                const float4v va = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(as, int(16 * ca), 0, 0));
                st[i] = c < xchunks ? vx : va;
            } else {
                st[i] = vx;
            }
        }
        if (prefetch) {
            load(0, b0);
            load(1, b1);
            load(2, b2);
        }
#pragma unroll
        for (int i = 0; i < kMvChunks; i++) {
            if (base + NT * i >= nchunks) break;
            const uint32_t c = base + tid + NT * i;
            if (c < nchunks) xl[c < xchunks ? xslot(c) : c] = st[i];
        }
    };
    stage_round(0, false);
    for (uint32_t base = NT * kMvChunks; base < nchunks; base += NT * kMvChunks) stage_round(base, false);
    float* part = reinterpret_cast<float*>(smem + 16 * nchunks);  // [4] wave partials
    __syncthreads();
    if constexpr (!LOOP) {
        load(0, b0);
        load(1, b1);
        load(2, b2);
    }
    if constexpr (PRO == kProRmsNorm) {
        // rmsnorm_kernel's arithmetic and order: its 256 threads' float4 sums strided by 1024
        // elements (the first four waves here), row sums, the four wave partials in fixed
        // order; then the elementwise rescale by every thread.
        if (tid < 256) {
            float ss = 0.f;
            for (uint32_t i = tid; i < xchunks; i += 256) {
                const float4v v = xl[xslot(i)];
                ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
            }
            ss = row16_sum(ss);
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            if (lane == 0) part[tid / 64] = ss;
        }
        __syncthreads();
        const float total = (part[0] + part[1]) + (part[2] + part[3]);
        const float scale = 1.0f / sqrtf(total / float(n_in) + a.eps);
        for (uint32_t i = tid; i < xchunks; i += NT) xl[xslot(i)] = xl[xslot(i)] * scale * xl[xchunks + i];
        __syncthreads();
    }

    float acc[RPH];
    auto compute = [&](uint32_t step, const uint32_t (&b)[RPH][NDW]) {
        const uint32_t c0 = step * 32 + l32;
        const uint32_t c = min(c0, last);
        float4v xv[8];
#pragma unroll
        for (int j = 0; j < 8; j++) xv[j] = xl[(c << 3) | (j ^ ((c >> 1) & 7))];
        float sx = 0.f, sx_hi = 0.f;
        if constexpr (T == kQ4_0 || T == kQ4_1 || T == kQ8_0) {
#pragma unroll
            for (int j = 0; j < 8; j++) sx += (xv[j][0] + xv[j][1]) + (xv[j][2] + xv[j][3]);
        } else if constexpr (T == kQ6_K) {  // the two 16-element halves separately
#pragma unroll
            for (int j = 0; j < 4; j++) sx += (xv[j][0] + xv[j][1]) + (xv[j][2] + xv[j][3]);
#pragma unroll
            for (int j = 4; j < 8; j++) sx_hi += (xv[j][0] + xv[j][1]) + (xv[j][2] + xv[j][3]);
        }
        const bool valid = c0 < ncols;
#pragma unroll
        for (int i = 0; i < RPH; i++) {
            // explicit roundings: every instantiation (rows per half-wave, prologue, epilogue)
            // sums a row in exactly the same way
            const float v = col_dot<T>(b[i], roff[i] + col_offset<T>(c), xv, sx, c, sx_hi);
            acc[i] = __fadd_rn(acc[i], valid ? v : 0.f);
        }
    };
    for (;;) {
    if constexpr (LOOP) {
        load(0, b0);
        load(1, b1);
        load(2, b2);
    }
#pragma unroll
    for (int i = 0; i < RPH; i++) acc[i] = 0.f;
    // three columns in flight (all of a 3072-long row), refilled as each is computed; the
    // last three buffered columns are computed without refills
    uint32_t st = 0;
    for (; st + 3 < nsteps; st += 3) {
        compute(st, b0);
        load(st + 3, b0);
        compute(st + 1, b1);
        load(st + 4, b1);
        compute(st + 2, b2);
        load(st + 5, b2);
    }
    compute(st, b0);
    compute(st + 1, b1);
    compute(st + 2, b2);

    // Row sums over the half-wave; lane i writes row i.
    float tot[RPH];
#pragma unroll
    for (int i = 0; i < RPH; i++) {
        float t = row16_sum(acc[i]);
        tot[i] = t + __shfl_xor(t, 16);
    }
    if constexpr (EPI == kEpiRopeKv) {
        // RPM is even and row0 + hw * RPM is even: each rotary pair is in one half-wave
        static_assert(RPM % 2 == 0, "rotary pairs stay in one half-wave");
        if (l32 < uint32_t(RPM)) {
            const uint32_t r = row0 + hw * RPM + l32;
            float val = tot[0];
#pragma unroll
            for (int i = 1; i < RPM; i++) val = l32 == uint32_t(i) ? tot[i] : val;
            if (m < 2) {
                // partner of the pair
                float x0 = tot[0], x1 = tot[1];
#pragma unroll
                for (int i = 2; i < RPM; i += 2) {
                    x0 = (l32 >> 1) == uint32_t(i / 2) ? tot[i] : x0;
                    x1 = (l32 >> 1) == uint32_t(i / 2) ? tot[i + 1] : x1;
                }
                const uint32_t pair = (r % a.head_dim) / 2;
                float sn, cs;
                sincosf(float(a.pos) * a.inv_freq[pair], &sn, &cs);
                val = (l32 & 1) ? rope_odd(x0, x1, cs, sn) : rope_even(x0, x1, cs, sn);
            }
            if (r < n_out) {
                if (m == 0) a.out[0][r] = val;
                else a.cache[m - 1][r] = _Float16(val);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < RPM; i++) {
            const uint32_t r = row0 + hw * RPM + i;
            if (l32 == uint32_t(i) && r < n_out) {
                float* o = a.out[m] + r;
                if constexpr (EPI == kEpiSiluGate) {
                    const float g = tot[i], u = tot[RPM + i];
                    *o = g / (1.0f + expf(-g)) * u;
                } else {
                    *o = EPI == kEpiAccumulate ? *o + tot[i] : tot[i];
                }
            }
        }
    }
    blk += gridDim.x;
    if (!LOOP || blk >= a.blocks) break;
    take_block();
    }
}

template <int T, int RPH, int PRO, int EPI, int NT, bool LOOP = false>
int launch_st(const MvArgs& a, uint32_t blocks, size_t lds, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&linear_stream_kernel<T, RPH, PRO, EPI, NT, LOOP>),
        hipFuncAttributeMaxDynamicSharedMemorySize, int(kMvLdsBytes));
    if (attr != hipSuccess) return -4;
    hipLaunchKernelGGL((linear_stream_kernel<T, RPH, PRO, EPI, NT, LOOP>), dim3(blocks), dim3(NT), lds, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <int T, int RPH, int PRO, int NT>
int launch_st_epi(const MvArgs& a, int epi, uint32_t blocks, size_t lds, hipStream_t stream) {
    switch (epi) {
        case kEpiStore:
            if constexpr (NT == 256 && Fmt<T>::blk > 1)
                if (blocks < a.blocks) return launch_st<T, RPH, PRO, kEpiStore, NT, true>(a, blocks, lds, stream);
            return launch_st<T, RPH, PRO, kEpiStore, NT>(a, blocks, lds, stream);
        case kEpiAccumulate: return launch_st<T, RPH, PRO, kEpiAccumulate, NT>(a, blocks, lds, stream);
        case kEpiRopeKv:
            if constexpr (RPH >= 2) return launch_st<T, RPH, PRO, kEpiRopeKv, NT>(a, blocks, lds, stream);
            return -2;
        default:
            if constexpr (RPH >= 2) return launch_st<T, RPH, PRO, kEpiSiluGate, NT>(a, blocks, lds, stream);
            return -2;
    }
}

// Workgroup shape: many rows per workgroup (x is staged once per workgroup, and its staging
// traffic otherwise rivals the weights' for the smaller matrices) while the grid still fills the
// 256 CUs: 512 threads with 4, 2 or 1 rows per half-wave when that gives 128..256 workgroups,
// else 256 threads with the most rows per half-wave that still gives >= 256 workgroups (the
// gate/up pair: at least 2, one of each matrix). F16/BF16 windows are 16 dwords: at most 2.
template <int T>
int launch_stream_t(MvArgs a, uint32_t n_mats, int pro, int epi, hipStream_t stream) {
    const bool silu = epi == kEpiSiluGate;
    // (Q6_K: 20-dword windows; two rows per half-wave only where an epilogue needs row pairs,
    // and then in 256-thread workgroups, whose register budget holds them without spilling)
    constexpr int kMaxRph = T == kQ6_K ? 1 : T == kF16 || T == kBF16 ? 2 : 4;
    const int min_rph = silu || epi == kEpiRopeKv ? 2 : 1;
    auto count = [&](int nt, int rph, bool set) {
        const uint32_t rpw = uint32_t(nt / 32) * uint32_t(silu ? rph / 2 : rph);  // rows per workgroup
        uint32_t blocks = 0;
        for (uint32_t m = 0; m < 3; m++) {
            if (m < n_mats && !(silu && m > 0)) blocks += (a.n_out[m] + rpw - 1) / rpw;
            if (set) a.blk_end[m] = blocks;
        }
        return blocks;
    };
    // (measured: a CU holds one 512-thread workgroup of this kernel at a time, so those are
    // used only when one round of at most 256 of them covers the rows)
    int nt = 0, rph = min_rph;
    for (int r = kMaxRph; r >= min_rph && !nt; r /= 2) {
        const uint32_t b = count(512, r, false);
        if (b >= 128 && b <= 256) { nt = 512; rph = r; }
    }
    for (int r = kMaxRph; r >= min_rph && !nt; r /= 2)
        if (count(256, r, false) >= 256 || r == min_rph) { nt = 256; rph = r; }
    if (!nt) { nt = 256; rph = min_rph; }  // (Q6_K pairs: min_rph above kMaxRph)
    a.blocks = count(nt, rph, true);
    // A block-quantized call of many more row blocks than the chip holds workgroups (a vocabulary; six
    // of 24 KB fit a CU, 1536 in all) loops over them: staging and normalizing x otherwise costs each
    // workgroup as much as its rows. Logits of 128256 x 3072 (rmsnorm), 16032 / 4008 blocks on 2048
    // workgroups: Q6_K 101.0 -> 82.9 us, Q4_0 56.0 -> 47.3, Q8_0 90.8 -> 80.1 (1024: 86.1, 48.3, 79.7;
    // 512: 95.8, 49.1, 82.5); F16 rows gain nothing (134.5, 136.0).
    constexpr uint32_t kLoopGrid = 2048;
    uint32_t blocks = a.blocks;
    if (Fmt<T>::blk > 1 && nt == 256 && epi == kEpiStore && blocks > kLoopGrid) {
        const uint32_t turns = (blocks + kLoopGrid - 1) / kLoopGrid;
        blocks = (blocks + turns - 1) / turns;
    }
    const size_t lds = size_t(a.n_in) * 4 * (pro == kProRmsNorm ? 2 : 1) + 16;
    if (lds > kMvLdsBytes) return -2;
    auto go = [&](auto pro_tag, auto nt_tag) -> int {
        constexpr int P = decltype(pro_tag)::value, N = decltype(nt_tag)::value;
        switch (rph) {
            case 4: if constexpr (kMaxRph >= 4) return launch_st_epi<T, 4, P, N>(a, epi, blocks, lds, stream); return -2;
            case 2: if constexpr (kMaxRph >= 2 || N == 256) return launch_st_epi<T, 2, P, N>(a, epi, blocks, lds, stream); return -2;
            default: return launch_st_epi<T, 1, P, N>(a, epi, blocks, lds, stream);
        }
    };
    using R = std::integral_constant<int, kProRmsNorm>;
    using X = std::integral_constant<int, kProNone>;
    using N5 = std::integral_constant<int, 512>;
    using N2 = std::integral_constant<int, 256>;
    if (pro == kProRmsNorm) return nt == 512 ? go(R{}, N5{}) : go(R{}, N2{});
    return nt == 512 ? go(X{}, N5{}) : go(X{}, N2{});
}

// Bytes of LDS a matvec workgroup stages (x, norm weights, rows) plus its reduction slots.
template <int T>
size_t matvec_lds(uint32_t n_in, uint32_t row_bytes, int R, int pro, int epi) {
    const int ns = epi == kEpiSiluGate ? 2 : 1;
    const size_t x = size_t(n_in) * 4 * (pro == kProRmsNorm ? 2 : 1);
    const size_t w = kMvStageW<T> ? (size_t(R) * row_bytes + 15 + 15) / 16 * 16 : 0;
    return x + ns * w + 4 * size_t(ns) * R * sizeof(float);
}

template <int T, int R, int PRO, int EPI>
int launch_mv(const MvArgs& a, uint32_t blocks, size_t lds, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&linear_matvec_kernel<T, R, PRO, EPI>),
        hipFuncAttributeMaxDynamicSharedMemorySize, int(kMvLdsBytes));
    if (attr != hipSuccess) return -4;
    hipLaunchKernelGGL((linear_matvec_kernel<T, R, PRO, EPI>), dim3(blocks), dim3(256), lds, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

template <int T, int R, int PRO>
int launch_mv_epi(const MvArgs& a, int epi, uint32_t blocks, size_t lds, hipStream_t stream) {
    switch (epi) {
        case kEpiStore: return launch_mv<T, R, PRO, kEpiStore>(a, blocks, lds, stream);
        case kEpiAccumulate: return launch_mv<T, R, PRO, kEpiAccumulate>(a, blocks, lds, stream);
        default:
            if constexpr (R <= 4) return launch_mv<T, R, PRO, kEpiSiluGate>(a, blocks, lds, stream);
            return -2;
    }
}

// One token through up to three matrices (n_mats) of type T: out[m] (+)= W[m]·x'.
template <int T>
int launch_matvec_t(MvArgs a, uint32_t n_mats, int pro, int epi, hipStream_t stream) {
    const uint32_t n_in = a.n_in;
    a.row_bytes = n_in / Fmt<T>::blk * Fmt<T>::bytes;
    if constexpr (kStreamed<T>) return launch_stream_t<T>(a, n_mats, pro, epi, stream);
    uint32_t rows = 0;
    for (uint32_t m = 0; m < n_mats; m++) rows = max(rows, a.n_out[m]);
    // Eight rows per matrix per workgroup when that still leaves >= 3 workgroups per CU
    // (measured: fewer, larger workgroups are slower here; more rows per workgroup only pay
    // for x traffic, which is not the limit) and the rows fit the staging buffer; four
    // otherwise. The gate/up pair takes four of each.
    // (One row per workgroup when four do not fit: long rows, e.g. a 28672-wide down projection.)
    int R = 4;
    if (epi != kEpiSiluGate && rows / 8 >= 768 && matvec_lds<T>(n_in, a.row_bytes, 8, pro, epi) <= kMvLdsBytes) R = 8;
    if (matvec_lds<T>(n_in, a.row_bytes, R, pro, epi) > kMvLdsBytes) R = 1;
    const size_t lds = matvec_lds<T>(n_in, a.row_bytes, R, pro, epi);
    if (lds > kMvLdsBytes) return -2;  // rows too long to stage
    uint32_t blocks = 0;
    for (uint32_t m = 0; m < 3; m++) {
        if (m < n_mats) blocks += (a.n_out[m] + R - 1) / R;
        a.blk_end[m] = blocks;
    }
    if (epi == kEpiSiluGate) blocks = a.blk_end[0];
    if (pro == kProRmsNorm)
        return R == 8 ? launch_mv_epi<T, 8, kProRmsNorm>(a, epi, blocks, lds, stream)
             : R == 4 ? launch_mv_epi<T, 4, kProRmsNorm>(a, epi, blocks, lds, stream)
                      : launch_mv_epi<T, 1, kProRmsNorm>(a, epi, blocks, lds, stream);
    return R == 8 ? launch_mv_epi<T, 8, kProNone>(a, epi, blocks, lds, stream)
         : R == 4 ? launch_mv_epi<T, 4, kProNone>(a, epi, blocks, lds, stream)
                  : launch_mv_epi<T, 1, kProNone>(a, epi, blocks, lds, stream);
}

// ---------------------------------------------------------------- several tokens

// The batched kernel is linear_tile.hip (one object per type); its shape is chosen here.
int launch_tile_type(uint32_t type, const TileCall& c) {
    switch (type) {
        case kF32:  return launch_tile<kF32>(c);
        case kF16:  return launch_tile<kF16>(c);
        case kBF16: return launch_tile<kBF16>(c);
        case kQ8_0: return launch_tile<kQ8_0>(c);
        case kQ4_0: return launch_tile<kQ4_0>(c);
        case kQ4_1: return launch_tile<kQ4_1>(c);
        case kQ6_K: return launch_tile<kQ6_K>(c);
        default:    return -2;
    }
}

template <int T>
int launch_t(const uint8_t* W, const float* x, float* out, uint32_t n_in, uint32_t n_out,
             uint32_t n_tok, uint32_t accumulate, uint32_t n_splits, void* workspace,
             size_t workspace_bytes, hipStream_t stream) {
    if (n_tok == 1) {
        MvArgs a{};
        a.W[0] = W;
        a.out[0] = out;
        a.n_out[0] = n_out;
        a.x = x;
        a.n_in = n_in;
        return launch_matvec_t<T>(a, 1, kProNone, accumulate ? kEpiAccumulate : kEpiStore, stream);
    }
    TileCall c{{W}, {out}, {n_out}, 1, x, n_in, n_tok, accumulate != 0, false,
               linear_shape(T, n_in, n_out, n_tok, workspace ? n_splits : 1, workspace_bytes), workspace, stream,
               workspace && n_splits != 1};
    return launch_tile<T>(c);
}

}  // namespace

uint32_t linear_splits(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t requested,
                       size_t workspace_bytes) {
    return n_tok <= 1 ? 1 : linear_shape(type, n_in, n_out, n_tok, requested, workspace_bytes).splits;
}

size_t linear_workspace_size(uint32_t type, uint32_t n_in, uint32_t n_out, uint32_t n_tok, uint32_t requested) {
    if (n_tok <= 1) return kLinearCounterBytes;
    const TileShape s = linear_shape(type, n_in, n_out, n_tok, requested, ~size_t(0));
    if (s.splits == 1) return kLinearCounterBytes;
    // (at least whole blocks of 256 rows x 64 tokens, so that the size does not depend on which
    // shape is the best for a few tokens more or less)
    const size_t blocks = (size_t(n_out) + 255) / 256 * ((size_t(n_tok) + 63) / 64) * 65536;
    return kLinearCounterBytes + s.splits * std::max(blocks, size_t(tile_count(n_out, n_tok, s)) * tile_bytes(s));
}

int launch_proj(uint32_t type, const void* const* W, const float* x, const float* aux,
                float* const* out, uint32_t n_in, const uint32_t* n_out, uint32_t n_mats,
                int pro, int epi, float eps, hipStream_t stream, const ProjRope* rope, uint32_t n_tok) {
    if (n_tok > 1) {  // a chunk: the batched kernel over every matrix's rows, no split-K
        // Epilogues: store, accumulate, or silu(gate) * up over two matrices (one launch with
        // gate and up rows paired in each tile).
        const bool pair = epi == kEpiSiluGate;
        if (pro != kProNone || rope) return -2;
        if (epi != kEpiStore && epi != kEpiAccumulate && !pair) return -2;
        if (pair && (n_mats != 2 || n_out[0] != n_out[1])) return -1;
        // (the matrices of each number of k groups in one launch: all of them, but for a mix of widths)
        for (uint32_t kg = 4; kg >= 1; kg /= 2) {
            TileCall c{};
            uint32_t rows = 0;
            for (uint32_t m = 0; m < n_mats; m++) {
                if (unsplit_k_groups(type, n_in, n_out[m], n_tok) != kg) continue;
                c.W[c.n_mats] = static_cast<const uint8_t*>(W[m]);
                c.out[c.n_mats] = pair ? out[0] : out[m];
                c.n_out[c.n_mats++] = n_out[m];
                rows += n_out[m];
            }
            if (rows == 0) continue;
            c.x = x;
            c.n_in = n_in;
            c.n_tok = n_tok;
            c.accumulate = epi == kEpiAccumulate;
            c.pair = pair;
            c.shape = unsplit_shape(type, n_in, rows, n_tok, kg);
            c.stream = stream;
            const int rc = launch_tile_type(type, c);
            if (rc != 0) return rc;
        }
        return 0;
    }
    MvArgs a{};
    if (epi == kEpiRopeKv) {
        if (!rope || n_mats != 3) return -2;
        if (!(type == kQ4_0 || type == kQ4_1 || type == kQ8_0 || type == kF16 || type == kBF16 || type == kQ6_K)) return -2;
        a.inv_freq = rope->inv_freq;
        a.cache[0] = rope->k_row;
        a.cache[1] = rope->v_row;
        a.head_dim = rope->head_dim;
        a.pos = rope->pos;
    }
    for (uint32_t m = 0; m < n_mats; m++) {
        a.W[m] = static_cast<const uint8_t*>(W[m]);
        a.n_out[m] = n_out[m];
        a.out[m] = epi == kEpiSiluGate || epi == kEpiRopeKv ? out[0] : out[m];
    }
    a.x = x;
    a.aux = aux;
    a.n_in = n_in;
    a.eps = eps;
    switch (type) {
        case kF32:  return launch_matvec_t<kF32>(a, n_mats, pro, epi, stream);
        case kF16:  return launch_matvec_t<kF16>(a, n_mats, pro, epi, stream);
        case kBF16: return launch_matvec_t<kBF16>(a, n_mats, pro, epi, stream);
        case kQ8_0: return launch_matvec_t<kQ8_0>(a, n_mats, pro, epi, stream);
        case kQ4_0: return launch_matvec_t<kQ4_0>(a, n_mats, pro, epi, stream);
        case kQ4_1: return launch_matvec_t<kQ4_1>(a, n_mats, pro, epi, stream);
        case kQ6_K: return launch_matvec_t<kQ6_K>(a, n_mats, pro, epi, stream);
        default:    return -2;
    }
}

int launch_linear(uint32_t type, const void* W, const float* x, float* out, uint32_t n_in,
                  uint32_t n_out, uint32_t n_tok, uint32_t accumulate, uint32_t n_splits,
                  void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const auto* w = static_cast<const uint8_t*>(W);
    switch (type) {
        case kF32:  return launch_t<kF32>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        case kF16:  return launch_t<kF16>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        case kBF16: return launch_t<kBF16>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        case kQ8_0: return launch_t<kQ8_0>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        case kQ4_0: return launch_t<kQ4_0>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        case kQ4_1: return launch_t<kQ4_1>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        case kQ6_K: return launch_t<kQ6_K>(w, x, out, n_in, n_out, n_tok, accumulate, n_splits, workspace, workspace_bytes, stream);
        default: return -2;
    }
}

}  // namespace ingot
