/* Decoding of the GGUF matrix formats outside the tuned Q4_K / IQ1_M / Q6_K
 * families: the codebooks and one lane's share of a 256-element super-block
 * (lane l of the reference's eight AVX2 lanes holds elements 32g + 4l .. +3 of
 * every group g), used by the GEMV kernels (q38_formats.hip) and the prompt
 * GEMM (q38_prompt.hip). */
#pragma once

#include "q38_device.h"
#include "q38_iq_grids.inc"

namespace q38 {

namespace {

/* ---- codebooks, expanded at compile time --------------------------------- */

#define Q38_IQ2_LEVEL(i) ((i) == 0 ? 8u : (i) == 1 ? 25u : 43u)
#define Q38_IQ2_BYTE(c, k) Q38_IQ2_LEVEL(((c) >> (2 * (k))) & 3)
#define Q38_IQ2_HALF(c, h) \
    (Q38_IQ2_BYTE(c, 4 * (h)) | Q38_IQ2_BYTE(c, 4 * (h) + 1) << 8 | Q38_IQ2_BYTE(c, 4 * (h) + 2) << 16 | \
     Q38_IQ2_BYTE(c, 4 * (h) + 3) << 24)
#define Q38_IQ2_ENTRY(c) Q38_IQ2_HALF(c, 0), Q38_IQ2_HALF(c, 1),
#define Q38_IQ3XXS_LEVEL(i) ((i) == 7 ? 62u : 8u * (i) + 4u)
#define Q38_IQ3XXS_ENTRY(c) \
    (Q38_IQ3XXS_LEVEL((c) & 7) | Q38_IQ3XXS_LEVEL(((c) >> 3) & 7) << 8 | Q38_IQ3XXS_LEVEL(((c) >> 6) & 7) << 16 | \
     Q38_IQ3XXS_LEVEL(((c) >> 9) & 7) << 24),
#define Q38_IQ3S_LEVEL(i) (2u * (i) + 1u)
#define Q38_IQ3S_ENTRY(c) \
    (Q38_IQ3S_LEVEL((c) & 7) | Q38_IQ3S_LEVEL(((c) >> 3) & 7) << 8 | Q38_IQ3S_LEVEL(((c) >> 6) & 7) << 16 | \
     Q38_IQ3S_LEVEL(((c) >> 9) & 7) << 24),

/* IQ2 grids: entry e, elements 4h..4h+3 at [2e + h]; IQ3 grids: entry e at [e] */
__device__ const uint32_t g_iq2xxs[512] = {Q38_IQ2XXS_CODES(Q38_IQ2_ENTRY)};
__device__ const uint32_t g_iq2xs[1024] = {Q38_IQ2XS_CODES(Q38_IQ2_ENTRY)};
__device__ const uint32_t g_iq2s[2048] = {Q38_IQ2S_CODES(Q38_IQ2_ENTRY)};
__device__ const uint32_t g_iq3xxs[256] = {Q38_IQ3XXS_CODES(Q38_IQ3XXS_ENTRY)};
__device__ const uint32_t g_iq3s[512] = {Q38_IQ3S_CODES(Q38_IQ3S_ENTRY)};

constexpr int8_t kIq4nl[16] = {Q38_IQ4NL_VALUES};
constexpr uint32_t pack4(int a, int b, int c, int d)
{
    return (uint32_t)(uint8_t)a | (uint32_t)(uint8_t)b << 8 | (uint32_t)(uint8_t)c << 16 | (uint32_t)(uint8_t)d << 24;
}
constexpr uint32_t kIq4nlT0 = pack4(kIq4nl[0], kIq4nl[1], kIq4nl[2], kIq4nl[3]);
constexpr uint32_t kIq4nlT1 = pack4(kIq4nl[4], kIq4nl[5], kIq4nl[6], kIq4nl[7]);
constexpr uint32_t kIq4nlT2 = pack4(kIq4nl[8], kIq4nl[9], kIq4nl[10], kIq4nl[11]);
constexpr uint32_t kIq4nlT3 = pack4(kIq4nl[12], kIq4nl[13], kIq4nl[14], kIq4nl[15]);

/* GGML type ids (include/qwen38/qwen38_gguf.h:29-52) */
enum : int {
    kF32 = 0, kF16 = 1, kQ4_0 = 2, kQ4_1 = 3, kQ5_0 = 6, kQ5_1 = 7, kQ8_0 = 8, kQ2K = 10, kQ3K = 11, kQ5K = 13,
    kIQ2XXS = 16, kIQ2XS = 17, kIQ3XXS = 18, kIQ1S = 19, kIQ4NL = 20, kIQ3S = 21, kIQ2S = 22, kIQ4XS = 23,
    kBF16 = 30
};

__device__ __forceinline__ uint32_t ld16(const uint8_t *p)
{
    return (uint32_t)p[0] | (uint32_t)p[1] << 8;
}
/* N dwords at a 2-byte aligned address (one load: the hardware takes
 * unaligned dwords) */
template <int N>
struct Dwords {
    uint32_t v[N];
};
template <int N>
__device__ __forceinline__ Dwords<N> ldn(const uint8_t *p)
{
    Dwords<N> r;
    __builtin_memcpy(&r, p, 4 * N);
    return r;
}
__device__ __forceinline__ uint32_t ld32u(const uint8_t *p) { return ldn<1>(p).v[0]; }
/* byte k of an array of dwords */
template <int N>
__device__ __forceinline__ uint32_t byte_of(const Dwords<N> &a, int k)
{
    return (a.v[k >> 2] >> (8 * (k & 3))) & 255u;
}
__device__ __forceinline__ uint32_t ld32a(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }

/* bytes of 0xff where bit k of `bits` (k < 4) is set */
__device__ __forceinline__ uint32_t byte_mask4(uint32_t bits)
{
    return ((bits & 15u) * 0x00204081u & 0x01010101u) * 0xffu;
}

/* negate the bytes selected by mask (values 1..127, so no byte borrows) */
__device__ __forceinline__ uint32_t negate_bytes(uint32_t v, uint32_t mask)
{
    return (v ^ mask) + (mask & 0x01010101u);
}

/* IQ2/IQ3 sign byte of a 7-bit index: even parity in bit 7 (ksigns_iq2xs) */
__device__ __forceinline__ uint32_t sign_byte(uint32_t index)
{
    index &= 127u;
    return index | (uint32_t)(__popc(index) & 1) << 7;
}

/* nibbles (one per byte) through the IQ4_NL table */
__device__ __forceinline__ uint32_t iq4nl_bytes(uint32_t nib)
{
    const uint32_t sel = nib & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(kIq4nlT1, kIq4nlT0, sel);
    const uint32_t hi = __builtin_amdgcn_perm(kIq4nlT3, kIq4nlT2, sel);
    const uint32_t high = ((nib >> 3) & 0x01010101u) * 0xffu;
    return (hi & high) | (lo & ~high);
}

__device__ __forceinline__ void k4_scale_min(int i, const uint8_t *p, int &sc, int &m)
{
    if (i < 4) {
        sc = p[i] & 63;
        m = p[i + 4] & 63;
    } else {
        sc = (p[i + 4] & 15) | ((p[i - 4] >> 6) << 4);
        m = (p[i + 4] >> 4) | ((p[i] >> 6) << 4);
    }
}

/* ---- Q8_K path: one lane's share of a super-block ------------------------- */

/* The lane's packed weights q[g] (elements 32g + 4l .. +3) and integer
 * scales s[g] of the eight groups, the block's scale factor before the
 * activation scale, and (Q2_K, Q5_K: dmin; IQ1_S: unused) the second
 * factor.  IQ4_NL keeps its eight group scales in gd[]. */
struct LaneBlock {
    uint32_t q[8];
    int s[8];
    float d, dmin;
    float gd[8];
};

template <int T>
constexpr uint32_t block_bytes()
{
    switch (T) {
    case kQ2K: return 84;
    case kQ3K: return 110;
    case kQ4K: return 144;
    case kQ5K: return 176;
    case kQ6K: return 210;
    case kIQ2XXS: return 66;
    case kIQ2XS: return 74;
    case kIQ2S: return 82;
    case kIQ3XXS: return 98;
    case kIQ3S: return 110;
    case kIQ4XS: return 136;
    case kIQ4NL: return 144;
    default: return 50;   /* IQ1_S */
    }
}

/* the 6-bit scales of the eight sub-blocks of Q4_K / Q5_K from the 12 packed
 * bytes, four per dword (sc) and the mins alike (m) (qwen38_quant.c:131-143) */
struct K4Scales {
    uint32_t sc[2], m[2];
};
__device__ __forceinline__ K4Scales k4_scales(const uint8_t *p)
{
    const Dwords<3> w = ldn<3>(p);
    return {{w.v[0] & 0x3f3f3f3fu, (w.v[2] & 0x0f0f0f0fu) | ((w.v[0] >> 2) & 0x30303030u)},
            {w.v[1] & 0x3f3f3f3fu, ((w.v[2] >> 4) & 0x0f0f0f0fu) | ((w.v[1] >> 2) & 0x30303030u)}};
}

/* the codebook of an IQ format as dwords: entries and their count (IQ1_S
 * takes the caller's table of 2048 x 8 int8) */
template <int T>
constexpr int table_dwords()
{
    switch (T) {
    case kIQ2XXS: return 512;
    case kIQ2XS: return 1024;
    case kIQ2S: return 2048;
    case kIQ3XXS: return 256;
    case kIQ3S: return 512;
    case kIQ1S: return 4096;
    default: return 0;
    }
}
template <int T>
__device__ __forceinline__ const uint32_t *table_of(const uint32_t *iq1s)
{
    if constexpr (T == kIQ2XXS) return g_iq2xxs;
    else if constexpr (T == kIQ2XS) return g_iq2xs;
    else if constexpr (T == kIQ2S) return g_iq2s;
    else if constexpr (T == kIQ3XXS) return g_iq3xxs;
    else if constexpr (T == kIQ3S) return g_iq3s;
    else return iq1s;
}

/* lane l's share of the block at blk; `table` is the format's codebook
 * (table_of, or a copy of it).  Header fields are loaded as whole dwords. */
template <int T>
__device__ __forceinline__ void decode_lane(const uint8_t *blk, int l, const uint32_t *table, LaneBlock &b)
{
    const int hi = l >= 4;
    if constexpr (T == kQ2K) {
        /* qwen38_quant.c:510-585 */
        const uint32_t d0 = ld32a(blk + 16 + 4 * l), d1 = ld32a(blk + 48 + 4 * l);
        const Dwords<4> sc = ldn<4>(blk);
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            b.q[g] = ((g < 4 ? d0 : d1) >> (2 * (g & 3))) & 0x03030303u;
            b.s[g] = (sc.v[g >> 1] >> (16 * (g & 1) + 8 * hi)) & 15;
        }
        const uint32_t dd = ld32a(blk + 80);
        b.d = f16_to_f32(dd);
        b.dmin = f16_to_f32(dd >> 16);
    } else if constexpr (T == kQ3K) {
        /* :587-662; scales :319-329: low nibbles of bytes 0..7, their high
         * nibbles, and two high bits each in bytes 8..11 */
        const uint32_t hm = ld32u(blk + 4 * l);
        const uint32_t d0 = ld32u(blk + 32 + 4 * l), d1 = ld32u(blk + 64 + 4 * l);
        const Dwords<3> sc = ldn<3>(blk + 96);
        const uint32_t six[4] = {(sc.v[0] & 0x0f0f0f0fu) | (sc.v[2] << 4 & 0x30303030u),
                                 (sc.v[1] & 0x0f0f0f0fu) | (sc.v[2] << 2 & 0x30303030u),
                                 (sc.v[0] >> 4 & 0x0f0f0f0fu) | (sc.v[2] & 0x30303030u),
                                 (sc.v[1] >> 4 & 0x0f0f0f0fu) | (sc.v[2] >> 2 & 0x30303030u)};
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t low = ((g < 4 ? d0 : d1) >> (2 * (g & 3))) & 0x03030303u;
            const uint32_t absent = ~(hm >> g) & 0x01010101u;
            b.q[g] = low + absent * 0xfcu;   /* minus 4 where the high bit is clear */
            b.s[g] = (int)((six[g >> 1] >> (16 * (g & 1) + 8 * hi)) & 63u) - 32;
        }
        b.d = f16_to_f32(ld16(blk + 108));
    } else if constexpr (T == kQ5K || T == kQ4K) {
        /* :1636-1725, :1546-1634 */
        const uint32_t qh = T == kQ5K ? ld32a(blk + 16 + 4 * l) : 0u;
        const K4Scales k4 = k4_scales(blk + 4);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t qs = ld32a(blk + (T == kQ5K ? 48 : 16) + 32 * c + 4 * l);
            b.q[2 * c] = qs & 0x0f0f0f0fu;
            b.q[2 * c + 1] = (qs >> 4) & 0x0f0f0f0fu;
            if constexpr (T == kQ5K) {
                b.q[2 * c] |= ((qh >> (2 * c)) & 0x01010101u) << 4;
                b.q[2 * c + 1] |= ((qh >> (2 * c + 1)) & 0x01010101u) << 4;
            }
        }
#pragma unroll
        for (int g = 0; g < 8; ++g) b.s[g] = (k4.sc[g >> 2] >> (8 * (g & 3))) & 255u;
        const uint32_t dd = ld32a(blk);
        b.d = f16_to_f32(dd);
        b.dmin = f16_to_f32(dd >> 16);
    } else if constexpr (T == kQ6K) {
        /* :1727-1814, the quants minus 32 (the reference's unsigned form
         * subtracts the 32s through the activation sums) */
        const Dwords<4> sc = ldn<4>(blk + 192);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t low[2] = {ld32u(blk + 64 * h + 4 * l), ld32u(blk + 64 * h + 32 + 4 * l)};
            const uint32_t high = ld32u(blk + 128 + 32 * h + 4 * l);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t v = ((low[j & 1] >> (j < 2 ? 0 : 4)) & 0x0f0f0f0fu) | ((high >> (2 * j)) & 0x03030303u) << 4;
                const uint32_t x = v ^ 0x20202020u;   /* 6-bit two's complement of v - 32 */
                b.q[4 * h + j] = x | ((x >> 5) & 0x01010101u) * 0xc0u;
                b.s[4 * h + j] = (int8_t)(sc.v[2 * h + (j >> 1)] >> (16 * (j & 1) + 8 * hi));
            }
        }
        b.d = f16_to_f32(ld16(blk + 208));
    } else if constexpr (T == kIQ2XXS) {
        /* :758-822 */
        const int sec = l >> 1, half = l & 1;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const Dwords<2> w = ldn<2>(blk + 2 + 8 * g);   /* four codes; sign indices and scale */
            const uint32_t grid = table[2 * ((w.v[0] >> (8 * sec)) & 255u) + half];
            const uint32_t signs = sign_byte(w.v[1] >> (7 * sec)) >> (4 * half);
            b.q[g] = negate_bytes(grid, byte_mask4(signs));
            b.s[g] = 1 + 2 * (int)(w.v[1] >> 28);
        }
        b.d = 0.125f * f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ2XS) {
        /* :824-893 */
        const int sec = l >> 1, half = l & 1;
        const Dwords<2> sc = ldn<2>(blk + 66);
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t code = ld16(blk + 2 + 8 * g + 2 * sec);
            const uint32_t grid = table[2 * (code & 511u) + half];
            b.q[g] = negate_bytes(grid, byte_mask4(sign_byte(code >> 9) >> (4 * half)));
            b.s[g] = 1 + 2 * (int)((sc.v[g >> 2] >> (8 * (g & 3) + 4 * hi)) & 15u);
        }
        b.d = 0.125f * f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ2S) {
        /* :664-756 */
        const int sec = l >> 1, half = l & 1;
        const Dwords<4> qh_sc = ldn<4>(blk + 66);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const Dwords<4> codes = ldn<4>(blk + 2 + 16 * p), sg = ldn<4>(blk + 34 + 16 * p);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int g = 4 * p + i;
                const uint32_t index = ((codes.v[i] >> (8 * sec)) & 255u) | ((byte_of(qh_sc, g) << (8 - 2 * sec)) & 0x300u);
                const uint32_t grid = table[2 * index + half];
                b.q[g] = negate_bytes(grid, byte_mask4(sg.v[i] >> (8 * sec + 4 * half)));
                b.s[g] = 1 + 2 * (int)((byte_of(qh_sc, 8 + g) >> (4 * hi)) & 15u);
            }
        }
        b.d = 0.125f * f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ3XXS) {
        /* :895-976 */
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const Dwords<4> meta = ldn<4>(blk + 66 + 16 * p);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int g = 4 * p + i;
                const uint32_t grid = table[blk[2 + 8 * g + l]];
                const uint32_t signs = sign_byte(meta.v[i] >> (7 * (l >> 1))) >> (4 * (l & 1));
                b.q[g] = negate_bytes(grid, byte_mask4(signs));
                b.s[g] = 1 + 2 * (int)(meta.v[i] >> 28);
            }
        }
        b.d = 0.25f * f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ3S) {
        /* :978-1061 */
        const Dwords<2> qh = ldn<2>(blk + 66);
        const uint32_t sc = ld32u(blk + 106);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const Dwords<4> sg = ldn<4>(blk + 74 + 16 * p);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int g = 4 * p + i;
                const uint32_t index = blk[2 + 8 * g + l] | (((byte_of(qh, g) >> l) & 1u) << 8);
                const uint32_t signs = sg.v[i] >> (8 * (l >> 1) + 4 * (l & 1));
                b.q[g] = negate_bytes(table[index], byte_mask4(signs));
                b.s[g] = 1 + 2 * (int)((sc >> (4 * g)) & 15u);
            }
        }
        b.d = f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ4XS) {
        /* :1063-1127 */
        const Dwords<2> head = ldn<2>(blk);   /* d, scale high bits; scale low nibbles */
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t qs = ld32a(blk + 8 + 16 * g + 4 * (l & 3));
            b.q[g] = iq4nl_bytes(hi ? qs >> 4 : qs);
            b.s[g] = (int)(((head.v[1] >> (4 * g)) & 15u) | ((head.v[0] >> (16 + 2 * g)) & 3u) << 4) - 32;
        }
        b.d = f16_to_f32(head.v[0]);
    } else if constexpr (T == kIQ4NL) {
        /* :1129-1175: eight 18-byte blocks */
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t qs = ld32u(blk + 18 * g + 2 + 4 * (l & 3));
            b.q[g] = iq4nl_bytes(hi ? qs >> 4 : qs);
            b.s[g] = 1;
            b.gd[g] = f16_to_f32(ld16(blk + 18 * g));
        }
    } else {
        /* IQ1_S, :1177-1253 */
        const int sec = l >> 1, half = l & 1;
        const Dwords<4> qh = ldn<4>(blk + 34);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const Dwords<4> codes = ldn<4>(blk + 2 + 16 * p);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int g = 4 * p + i;
                const uint32_t high = (qh.v[g >> 1] >> (16 * (g & 1))) & 0xffffu;
                const uint32_t index = ((codes.v[i] >> (8 * sec)) & 255u) | (((high >> (3 * sec)) & 7u) << 8);
                b.q[g] = table[2 * index + half];
                b.s[g] = 1 + 2 * (int)((high >> 12) & 7u);
            }
        }
        b.d = f16_to_f32(ld16(blk));
    }
}

/* the multipliers of activation sums 2l and 2l + 1 of a block in its integer
 * min (Q2_K, Q5_K) or correction (IQ1_S) sum */
template <int T>
__device__ __forceinline__ void extra_factors(const uint8_t *blk, int l, int &m0, int &m1)
{
    if constexpr (T == kQ2K) {
        const uint32_t w = ld16(blk + 2 * l);
        m0 = (w >> 4) & 15;
        m1 = w >> 12;
    } else if constexpr (T == kIQ1S) {
        const uint32_t high = ld16(blk + 34 + 2 * l);
        const int scale = 1 + 2 * (int)((high >> 12) & 7u);
        m0 = m1 = high & 0x8000u ? -scale : scale;
    } else {
        const K4Scales k4 = k4_scales(blk + 4);
        m0 = m1 = (int)(((l < 4 ? k4.m[0] : k4.m[1]) >> (8 * (l & 3))) & 255u);
    }
}

__device__ __forceinline__ float bf16_to_f32(uint32_t bits) { return __uint_as_float(bits << 16); }

/* The weight expression of element i of a block (the first operand of its
 * fmaf in the float dot), i < elements per block. */
template <int T>
__device__ __forceinline__ float element_weight(const uint8_t *blk, int i)
{
    if constexpr (T == kQ8_0) {
        return __fmul_rn(f16_to_f32(ld16(blk)), (float)(int8_t)blk[2 + i]);
    } else if constexpr (T == kIQ4NL) {
        const uint32_t byte = blk[2 + (i & 15)];
        return __fmul_rn(f16_to_f32(ld16(blk)), (float)kIq4nl[i < 16 ? byte & 15 : byte >> 4]);
    } else if constexpr (T == kQ2K) {
        const int s = i / 16, j = i % 16, half = s / 8, field = (s % 8) / 2, part = s % 2;
        const float scale = __fmul_rn(f16_to_f32(ld16(blk + 80)), (float)(blk[s] & 15));
        const float minimum = __fmul_rn(f16_to_f32(ld16(blk + 82)), (float)(blk[s] >> 4));
        const int q = (blk[16 + 32 * half + 16 * part + j] >> (2 * field)) & 3;
        return __fsub_rn(__fmul_rn(scale, (float)q), minimum);
    } else if constexpr (T == kQ3K) {
        const int g = i / 32, j = i % 32, half = g / 4, field = g % 4, si = 2 * g + j / 16;
        const uint8_t *sc = blk + 96;
        const int s = ((si < 8 ? sc[si] & 15 : sc[si - 8] >> 4) | (((sc[8 + si % 4] >> (2 * (si / 4))) & 3) << 4)) - 32;
        const int q = ((blk[32 + 32 * half + j] >> (2 * field)) & 3) - ((blk[j] >> g) & 1 ? 0 : 4);
        return __fmul_rn(__fmul_rn(f16_to_f32(ld16(blk + 108)), (float)s), (float)q);
    } else if constexpr (T == kQ4K || T == kQ5K) {
        constexpr bool five = T == kQ5K;
        const int c = i / 64, upper = (i % 64) / 32, j = i % 32;
        int sc, m;
        k4_scale_min(2 * c + upper, blk + 4, sc, m);
        const uint8_t byte = blk[(five ? 48 : 16) + 32 * c + j];
        int q = upper ? byte >> 4 : byte & 15;
        if (five && ((blk[16 + j] >> (2 * c + upper)) & 1)) q += 16;
        const float dd = __fmul_rn(f16_to_f32(ld16(blk)), (float)sc);
        const float mm = __fmul_rn(f16_to_f32(ld16(blk + 2)), (float)m);
        return __fsub_rn(__fmul_rn(dd, (float)q), mm);
    } else {
        /* Q6_K: element 128 half + 32 k + i0 */
        const int half = i / 128, k = (i % 128) / 32, i0 = i % 32;
        const uint8_t *ql = blk + 64 * half, *qh = blk + 128 + 32 * half;
        const uint8_t lowb = ql[i0 + (k & 1) * 32];
        const int q = ((k < 2 ? lowb & 15 : lowb >> 4) | (((qh[i0] >> (2 * k)) & 3) << 4)) - 32;
        const float ds = __fmul_rn(f16_to_f32(ld16(blk + 208)), (float)reinterpret_cast<const int8_t *>(blk + 192)[8 * half + i0 / 16 + 2 * k]);
        return __fmul_rn(ds, (float)q);
    }
}

template <int T>
constexpr bool has_extra()
{
    return T == kQ2K || T == kQ5K || T == kIQ1S;
}

}  // namespace

}  // namespace q38
