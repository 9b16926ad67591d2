/* Matrices against fp32 activations (q38_tensor_gemv_f32 / gemm_f32,
 * src/qwen38/qwen38_quant.c:2812-2831, 2924-2948): F32, F16, BF16, Q8_0 and,
 * through the same entry points, IQ4_NL and the K-quants.
 *
 * Arithmetic (q38_dot_row, :2768-2810): per (row, token) one chain
 * total = fmaf(w_e, x_e, total) over the row's elements in the reference's
 * order, each weight expression rounded as the reference rounds it.  The
 * order is the element order but for IQ4_NL (elements j and 16 + j of a block
 * alternate) and Q6_K (elements i, 32 + i, 64 + i, 96 + i of a half block).
 *
 * Split.  The chain is serial, so one token of a row takes at least `width`
 * dependent fmas (6 cycles each on one wavefront: 13 us for 5120 columns, 44
 * us for 17408) and what can be taken off it runs elsewhere.  A workgroup has
 * 64 rows: chain wavefronts hold one row per lane and MT tokens each, four
 * producer wavefronts load the rows with 16 consecutive lanes on one row,
 * form the weights and leave them in LDS as fp32, 64 columns per stage, next
 * to the stage's activations.  A chain wavefront reads 16 columns of its row
 * with four 16-byte LDS reads, a group ahead of their use, and takes each
 * activation by a DPP row broadcast inside the fma, so a link is one
 * instruction.  Two LDS slots: at barrier k stage k + 1 is complete and the
 * last columns of stage k have been read, so its slot takes stage k + 2.  The
 * producers keep kAhead stages of loads in registers: a quad's own header
 * fields and quant bytes, from which its four weights are formed when the stage
 * is stored (decoding element by element from memory at that point, a Q4_K
 * matrix of 5120 x 5120, one token, took 320 us and one of 65536 x 768 165; 56
 * and 25 now).
 *
 * Bound.  One token: the chain on matrices of up to 16384 rows, HBM on taller
 * ones (F32 34816 x 5120 148 us, 4.8 TB/s; F16 78 us, 4.6 TB/s).  One thread
 * per row reading its own elements took 778 and 725 us there, 2342 us on F16
 * 5120 x 17408 (now 91), 442 us on F32 96 x 5120 (now 24) and 446 us on Q8_0
 * 5120 x 17408 (now 99).  Prompts: fma issue, 64 tokens x 34816 x 5120 482 us
 * (F16; launches of four tokens took 12.3 ms).  Measured and dropped: plain
 * fmas with the activation broadcast by LDS reads (one token 43 against 31
 * us: twice the LDS reads), one group of columns ahead instead of two for
 * one token (31 against 29 us).
 */
#include "q38_format_decode.h"
#include "q38_kernels.h"

#include <type_traits>

namespace q38 {

namespace {

constexpr int kFloatRows = 64;
constexpr int kProducers = 256;
/* one quad of columns of the 64 rows, 16 bytes apart from the next bank group */
constexpr int kQuadBytes = kFloatRows * 16 + 16;

/* matrix column of chain position c */
template <int T>
__device__ __forceinline__ uint32_t chain_column(uint32_t c)
{
    if constexpr (T == kIQ4NL) return (c & ~31u) | (c & 1u) << 4 | ((c >> 1) & 15u);
    else if constexpr (T == kQ6K) return (c & ~127u) | (c & 3u) << 5 | ((c >> 2) & 31u);
    else return c;
}

/* four consecutive chain positions of one row: what is loaded ahead, and the
 * weights it gives, each the expression element_weight has.  Positions past the
 * width load nothing and give values that no chain reads. */
template <int T>
struct QuadLoad;
/* signed bytes of v as floats times s */
__device__ __forceinline__ float4 scaled_bytes(float s, uint32_t v)
{
    return make_float4(fmul_rn(s, (float)(int8_t)v), fmul_rn(s, (float)(int8_t)(v >> 8)),
                       fmul_rn(s, (float)(int8_t)(v >> 16)), fmul_rn(s, (float)((int32_t)v >> 24)));
}
/* s * q - m for the bytes q of v */
__device__ __forceinline__ float4 scaled_minus(float s, uint32_t v, float m)
{
    return make_float4(__fsub_rn(fmul_rn(s, (float)(v & 255u)), m), __fsub_rn(fmul_rn(s, (float)(v >> 8 & 255u)), m),
                       __fsub_rn(fmul_rn(s, (float)(v >> 16 & 255u)), m), __fsub_rn(fmul_rn(s, (float)(v >> 24)), m));
}
template <>
struct QuadLoad<kF32> {
    float v[4];
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t width)
    {
        const uint8_t *p = row + 4 * (size_t)c;
        if (!Edge || c + 3 < width) __builtin_memcpy(v, p, 16);
        else
            for (int k = 0; k < 4; ++k) v[k] = c + k < width ? *reinterpret_cast<const float *>(p + 4 * k) : 0.0f;
    }
    __device__ __forceinline__ float4 weights(uint32_t) const
    {
        return make_float4(v[0], v[1], v[2], v[3]);
    }
};
template <int T>
struct QuadLoad16 {
    uint32_t v[2];
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t width)
    {
        const uint8_t *p = row + 2 * (size_t)c;
        if (!Edge || c + 3 < width) {
            __builtin_memcpy(v, p, 8);
        } else {
            uint32_t h[4];
            for (int k = 0; k < 4; ++k) h[k] = c + k < width ? ld16(p + 2 * k) : 0u;
            v[0] = h[0] | h[1] << 16;
            v[1] = h[2] | h[3] << 16;
        }
    }
    __device__ __forceinline__ float4 weights(uint32_t) const
    {
        if constexpr (T == kF16)
            return make_float4(f16_to_f32(v[0]), f16_to_f32(v[0] >> 16), f16_to_f32(v[1]), f16_to_f32(v[1] >> 16));
        else
            return make_float4(bf16_to_f32(v[0]), __uint_as_float(v[0] & 0xffff0000u), bf16_to_f32(v[1]),
                               __uint_as_float(v[1] & 0xffff0000u));
    }
};
template <> struct QuadLoad<kF16> : QuadLoad16<kF16> {};
template <> struct QuadLoad<kBF16> : QuadLoad16<kBF16> {};
template <>
struct QuadLoad<kQ8_0> {
    uint32_t q, d;
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t width)
    {
        if (Edge) q = d = 0;
        if (!Edge || c < width) {   /* a multiple of 32 */
            const uint8_t *blk = row + (size_t)(c / 32) * 34;
            d = ld16(blk);
            __builtin_memcpy(&q, blk + 2 + c % 32, 4);
        }
    }
    __device__ __forceinline__ float4 weights(uint32_t) const
    {
        return scaled_bytes(f16_to_f32(d), q);
    }
};

/* IQ4_NL: positions 2j, 2j + 1 are elements j and 16 + j, so a quad is two bytes */
template <>
struct QuadLoad<kIQ4NL> {
    uint32_t q, d;
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t width)
    {
        if (Edge) q = d = 0;
        if (!Edge || c < width) {   /* a multiple of 32 */
            const uint8_t *blk = row + (size_t)(c / 32) * 18;
            d = ld16(blk);
            q = ld16(blk + 2 + c % 32 / 2);
        }
    }
    __device__ __forceinline__ float4 weights(uint32_t) const
    {
        return scaled_bytes(f16_to_f32(d), iq4nl_bytes((q & 15u) | (q << 4 & 0xf00u) | (q << 8 & 0xf0000u) | (q << 12 & 0xf000000u)));
    }
};
/* the K-quants' widths are multiples of 256: no stage ends inside a block */
template <>
struct QuadLoad<kQ2K> {
    uint32_t q, dd, sc;
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t)
    {
        const uint8_t *blk = row + (size_t)(c / 256) * 84;
        const uint32_t i = c % 256;   /* half i / 128, field i / 32 % 4, byte i % 32 */
        __builtin_memcpy(&q, blk + 16 + (i / 128) * 32 + i % 32, 4);
        __builtin_memcpy(&dd, blk + 80, 4);
        sc = blk[i / 16];
    }
    __device__ __forceinline__ float4 weights(uint32_t c) const
    {
        return scaled_minus(fmul_rn(f16_to_f32(dd), (float)(sc & 15u)), (q >> (c % 128 / 32 * 2)) & 0x03030303u,
                            fmul_rn(f16_to_f32(dd >> 16), (float)(sc >> 4)));
    }
};
template <>
struct QuadLoad<kQ3K> {
    uint32_t q, high, sc, sc_high, d;
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t)
    {
        const uint8_t *blk = row + (size_t)(c / 256) * 110;
        const uint32_t i = c % 256, s = i / 16;
        __builtin_memcpy(&q, blk + 32 + (i / 128) * 32 + i % 32, 4);
        __builtin_memcpy(&high, blk + i % 32, 4);
        sc = blk[96 + s % 8];
        sc_high = blk[104 + s % 4];
        d = ld16(blk + 108);
    }
    __device__ __forceinline__ float4 weights(uint32_t c) const
    {
        const uint32_t i = c % 256, s = i / 16;
        const int scale = (int)((sc >> (s / 8 * 4) & 15u) | (sc_high >> (s / 4 * 2) & 3u) << 4) - 32;
        const uint32_t absent = ~(high >> (i / 32)) & 0x01010101u;   /* minus 4 where the high bit is clear */
        return scaled_bytes(fmul_rn(f16_to_f32(d), (float)scale),
                            ((q >> (c % 128 / 32 * 2)) & 0x03030303u) + absent * 0xfcu);
    }
};
template <int T>
struct QuadLoadK45 {
    uint32_t head[4], q, high;   /* d and dmin, twelve scale bytes; quants */
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t)
    {
        const uint8_t *blk = row + (size_t)(c / 256) * (T == kQ5K ? 176 : 144);
        const uint32_t i = c % 256;
        __builtin_memcpy(head, blk, 16);
        __builtin_memcpy(&q, blk + (T == kQ5K ? 48 : 16) + i / 64 * 32 + i % 32, 4);
        if (T == kQ5K) __builtin_memcpy(&high, blk + 16 + i % 32, 4);
    }
    __device__ __forceinline__ float4 weights(uint32_t c) const
    {
        const uint32_t s = c % 256 / 32, at = s % 4 * 8;
        const uint32_t sc = s < 4 ? head[1] & 0x3f3f3f3fu : (head[3] & 0x0f0f0f0fu) | (head[1] >> 2 & 0x30303030u);
        const uint32_t m = s < 4 ? head[2] & 0x3f3f3f3fu : (head[3] >> 4 & 0x0f0f0f0fu) | (head[2] >> 2 & 0x30303030u);
        uint32_t v = (q >> (s % 2 * 4)) & 0x0f0f0f0fu;
        if (T == kQ5K) v |= (high >> s & 0x01010101u) << 4;
        return scaled_minus(fmul_rn(f16_to_f32(head[0]), (float)(sc >> at & 255u)), v,
                            fmul_rn(f16_to_f32(head[0] >> 16), (float)(m >> at & 255u)));
    }
};
template <> struct QuadLoad<kQ4K> : QuadLoadK45<kQ4K> {};
template <> struct QuadLoad<kQ5K> : QuadLoadK45<kQ5K> {};
/* Q6_K: positions 4j .. 4j + 3 of a half block are elements j, 32 + j, 64 + j
 * and 96 + j: two quant bytes, one byte of their high bits, every second scale */
template <>
struct QuadLoad<kQ6K> {
    uint32_t low, low32, high, sc[2], d;
    template <bool Edge>
    __device__ __forceinline__ void load(const uint8_t *row, uint32_t c, uint32_t)
    {
        const uint8_t *blk = row + (size_t)(c / 256) * 210;
        const uint32_t half = c % 256 / 128, j = c % 128 / 4;
        low = blk[64 * half + j];
        low32 = blk[64 * half + 32 + j];
        high = blk[128 + 32 * half + j];
        __builtin_memcpy(sc, blk + 192 + 8 * half, 8);
        d = ld16(blk + 208);
    }
    __device__ __forceinline__ float4 weights(uint32_t c) const
    {
        const uint32_t at = c % 128 / 64 * 8;   /* scales 0, 2, 4, 6 or 1, 3, 5, 7 of the half */
        const float dv = f16_to_f32(d);
        auto weight = [&](uint32_t nibble, int k) {
            const int q = (int)((nibble & 15u) | (high >> (2 * k) & 3u) << 4) - 32;
            const int s = (int8_t)(sc[k / 2] >> (16 * (k % 2) + at));
            return fmul_rn(fmul_rn(dv, (float)s), (float)q);
        };
        return make_float4(weight(low, 0), weight(low32, 1), weight(low >> 4, 2), weight(low32 >> 4, 3));
    }
};

/* the 16 links of a group for N tokens: a[t] = fmaf(x of column k, w[k],
 * a[t]), x[t] of lane k of each 16-lane row being column k's activation.  The
 * tokens alternate, so their chains fill each other's latency.  One
 * statement, opening with the two wait states a DPP read of a VGPR written by
 * the VALU just before needs. */
#define Q38_TAIL " row_mask:0xf bank_mask:0xf\n\t"
#define Q38_LINK1(w, n) "v_fmac_f32_dpp %0, %1, %" #w " row_newbcast:" #n Q38_TAIL
#define Q38_LINK2(w, n) \
    "v_fmac_f32_dpp %0, %2, %" #w " row_newbcast:" #n Q38_TAIL "v_fmac_f32_dpp %1, %3, %" #w " row_newbcast:" #n Q38_TAIL
#define Q38_LINK4(w, n)                                                                                            \
    "v_fmac_f32_dpp %0, %4, %" #w " row_newbcast:" #n Q38_TAIL "v_fmac_f32_dpp %1, %5, %" #w " row_newbcast:" #n Q38_TAIL \
    "v_fmac_f32_dpp %2, %6, %" #w " row_newbcast:" #n Q38_TAIL "v_fmac_f32_dpp %3, %7, %" #w " row_newbcast:" #n Q38_TAIL
#define Q38_W(w) \
    "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), \
        "v"(w[10]), "v"(w[11]), "v"(w[12]), "v"(w[13]), "v"(w[14]), "v"(w[15])

__device__ __forceinline__ void links1(float &a, float x, const float (&w)[16])
{
    asm volatile("s_nop 1\n\t" Q38_LINK1(2, 0) Q38_LINK1(3, 1) Q38_LINK1(4, 2) Q38_LINK1(5, 3) Q38_LINK1(6, 4)
                     Q38_LINK1(7, 5) Q38_LINK1(8, 6) Q38_LINK1(9, 7) Q38_LINK1(10, 8) Q38_LINK1(11, 9)
                         Q38_LINK1(12, 10) Q38_LINK1(13, 11) Q38_LINK1(14, 12) Q38_LINK1(15, 13) Q38_LINK1(16, 14)
                             Q38_LINK1(17, 15)
                 : "+v"(a) : "v"(x), Q38_W(w));
}
__device__ __forceinline__ void links2(float &a, float &b, float x, float y, const float (&w)[16])
{
    asm volatile("s_nop 1\n\t" Q38_LINK2(4, 0) Q38_LINK2(5, 1) Q38_LINK2(6, 2) Q38_LINK2(7, 3) Q38_LINK2(8, 4)
                     Q38_LINK2(9, 5) Q38_LINK2(10, 6) Q38_LINK2(11, 7) Q38_LINK2(12, 8) Q38_LINK2(13, 9)
                         Q38_LINK2(14, 10) Q38_LINK2(15, 11) Q38_LINK2(16, 12) Q38_LINK2(17, 13) Q38_LINK2(18, 14)
                             Q38_LINK2(19, 15)
                 : "+v"(a), "+v"(b) : "v"(x), "v"(y), Q38_W(w));
}
__device__ __forceinline__ void links4(float &a, float &b, float &c, float &d, float x, float y, float z, float u,
                                       const float (&w)[16])
{
    asm volatile("s_nop 1\n\t" Q38_LINK4(8, 0) Q38_LINK4(9, 1) Q38_LINK4(10, 2) Q38_LINK4(11, 3) Q38_LINK4(12, 4)
                     Q38_LINK4(13, 5) Q38_LINK4(14, 6) Q38_LINK4(15, 7) Q38_LINK4(16, 8) Q38_LINK4(17, 9)
                         Q38_LINK4(18, 10) Q38_LINK4(19, 11) Q38_LINK4(20, 12) Q38_LINK4(21, 13) Q38_LINK4(22, 14)
                             Q38_LINK4(23, 15)
                 : "+v"(a), "+v"(b), "+v"(c), "+v"(d) : "v"(x), "v"(y), "v"(z), "v"(u), Q38_W(w));
}
/* LDS traffic of the stage done, then the barrier; global loads stay in flight */
__device__ __forceinline__ void stage_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

/* 16 columns of a lane's row, and the wavefront's tokens' activations of
 * column lane % 16 */
template <int MT>
struct Group {
    float w[16], x[MT];

    __device__ __forceinline__ void read(const uint8_t *slot, const float *xs, int stage, int group, int lane)
    {
#pragma unroll
        for (int t = 0; t < MT; ++t) x[t] = xs[t * stage + 16 * group + (lane & 15)];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float4 v = *reinterpret_cast<const float4 *>(slot + (4 * group + k) * kQuadBytes + lane * 16);
            w[4 * k] = v.x;
            w[4 * k + 1] = v.y;
            w[4 * k + 2] = v.z;
            w[4 * k + 3] = v.w;
        }
    }
    __device__ __forceinline__ void links(float (&a)[MT]) const
    {
        constexpr int kFours = MT / 4 * 4;
#pragma unroll
        for (int t = 0; t < kFours; t += 4)
            links4(a[t], a[t + 1], a[t + 2], a[t + 3], x[t], x[t + 1], x[t + 2], x[t + 3], w);
        if constexpr (MT % 4 >= 2) links2(a[kFours], a[kFours + 1], x[kFours], x[kFours + 1], w);
        if constexpr (MT % 2) links1(a[MT - 1], x[MT - 1], w);
    }
};

/* stages that hold `width` columns, up to the widest row an entry point takes.
 * The host passes the count: worked out in the kernel this way, the compiler
 * orders the producers' loads differently and eight tokens take longer (F16
 * 5120 x 6144 121 against 104 us). */
constexpr int stages_of(uint32_t width, uint32_t stage) { return (int)((width - 1) / stage + 1); }
static_assert(stages_of(1, 64) == 1 && stages_of(64, 64) == 1 && stages_of(65, 64) == 2 &&
                  stages_of(0xffffffffu, 64) == 1 << 26 && stages_of(0xffffffffu, 128) == 1 << 25,
              "stages");

/* quads of five dwords and more: one stage less in registers */
template <int T>
constexpr bool kWideQuad = sizeof(QuadLoad<T>) > 16;

/* y[t * ldy + row]: 64 rows, MT tokens in each of CW chain wavefronts, stages
 * of ST columns */
template <int T, int MT, int CW, int ST>
__global__ __launch_bounds__(64 * CW + kProducers, ST == 128 ? 2 : CW == 1 && !kWideQuad<T> ? 5 : 4) void gemm_float_kernel(const uint8_t *__restrict__ w,
                                                                        const float *__restrict__ x,
                                                                        float *__restrict__ y, uint32_t ldy,
                                                                        uint32_t rows, uint32_t width,
                                                                        uint32_t row_bytes, uint32_t tokens, int stages)
{
    constexpr int kTok = MT * CW;
    constexpr int kFloatStage = ST, kFloatQuads = ST / 4, kGroups = ST / 16, kSlotBytes = kFloatQuads * kQuadBytes;
    constexpr int kAhead = kTok > 16 || kWideQuad<T> ? 2 : 3;
    constexpr int kWItems = kFloatRows * kFloatQuads / kProducers;
    constexpr int kXItems = (kTok * kFloatQuads + kProducers - 1) / kProducers;
    constexpr int kXSlot = kTok * kFloatStage * 4;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * (kSlotBytes + kXSlot)];
    const uint32_t row0 = blockIdx.x * kFloatRows, tok0 = blockIdx.y * kTok;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    if (wave >= CW) {
        /* ---- producers ---- */
        const int tid = (int)threadIdx.x - 64 * CW;
        struct Stage {
            QuadLoad<T> w[kWItems];
            float4 x[kXItems];
        } ring[kAhead];
        const uint8_t *wbase = w + (size_t)row0 * row_bytes;
        uint32_t wrow[kWItems];   /* byte offsets of the rows (rows past the matrix repeat the last one) */
#pragma unroll
        for (int k = 0; k < kWItems; ++k) {
            const uint32_t r = (tid + k * kProducers) / kFloatQuads, have = rows - row0 - 1;
            wrow[k] = (r < have ? r : have) * row_bytes;
        }
        const uint32_t quad = 4 * (tid % kFloatQuads);   /* the same in every item */
        static_assert(kProducers % kFloatQuads == 0, "one column quad per thread");
        /* Edge: the stage may end past the width.  Other stages load without
         * a branch, which the compiler answers by waiting for every load in
         * flight. */
        auto load = [&](auto edge, Stage &s, int stage) {
            constexpr bool Edge = decltype(edge)::value;
            const uint32_t c = (uint32_t)stage * kFloatStage + quad;
#pragma unroll
            for (int k = 0; k < kWItems; ++k) s.w[k].template load<Edge>(wbase + wrow[k], c, width);
#pragma unroll
            for (int k = 0; k < kXItems; ++k) {
                const int t = (tid + k * kProducers) / kFloatQuads;
                const uint32_t tok = tok0 + (t < kTok ? t : kTok - 1);
                const float *xr = x + (size_t)(tok < tokens ? tok : tokens - 1) * width;
                if (chain_column<T>(1) == 1 && (!Edge || c + 3 < width)) {
                    __builtin_memcpy(&s.x[k], xr + c, 16);
                } else {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = !Edge || c + e < width ? xr[chain_column<T>(c + e)] : 0.0f;
                    s.x[k] = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        };
        auto store = [&](const Stage &s, int stage) {
            uint8_t *slot = lds + (stage & 1) * (kSlotBytes + kXSlot);
            const uint32_t c = (uint32_t)stage * kFloatStage + quad;
#pragma unroll
            for (int k = 0; k < kWItems; ++k) {
                const int r = (tid + k * kProducers) / kFloatQuads;
                *reinterpret_cast<float4 *>(slot + (quad / 4) * kQuadBytes + r * 16) = s.w[k].weights(c);
            }
#pragma unroll
            for (int k = 0; k < kXItems; ++k) {
                const int t = (tid + k * kProducers) / kFloatQuads;
                if (t < kTok) *reinterpret_cast<float4 *>(slot + kSlotBytes + (t * kFloatStage + quad) * 4) = s.x[k];
            }
        };
        const int full = (int)(width / kFloatStage);
        auto load_any = [&](Stage &s, int stage) {
            if (stage < full) load(std::false_type(), s, stage);
            else if (stage < stages) load(std::true_type(), s, stage);
        };
#pragma unroll
        for (int i = 0; i < kAhead; ++i) load_any(ring[i], i);
        int s0 = 0;
#pragma unroll 1
        for (; s0 + 2 * kAhead <= full; s0 += kAhead) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
                store(ring[i], s0 + i);
                load(std::false_type(), ring[i], s0 + i + kAhead);
                stage_barrier();
            }
        }
#pragma unroll 1
        for (; s0 < stages; s0 += kAhead) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
                if (s0 + i < stages) {
                    store(ring[i], s0 + i);
                    load_any(ring[i], s0 + i + kAhead);
                    stage_barrier();
                }
            }
        }
        stage_barrier();
        return;
    }

    /* ---- chains ---- */
    const int lane = threadIdx.x & 63;
    __builtin_amdgcn_s_setprio(3);
    float acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = 0.0f;
    auto slot_of = [&](int stage) { return lds + (stage & 1) * (kSlotBytes + kXSlot); };
    auto read = [&](Group<MT> &g, const uint8_t *slot, int group) {
        g.read(slot, reinterpret_cast<const float *>(slot + kSlotBytes) + wave * MT * kFloatStage, kFloatStage, group, lane);
    };
    const int full = (int)(width / kFloatStage), rest = (int)(width % kFloatStage);
    stage_barrier();   /* stage 0 is there */
    /* one to three tokens: a group's links take about 100 cycles, less than
     * the LDS reads of one, so two groups are in flight */
    if constexpr (MT <= 3) {
        Group<MT> g[4];
        if (full) {
            read(g[0], slot_of(0), 0);
            read(g[1], slot_of(0), 1);
        }
#pragma unroll 1
        for (int s = 0; s < full; ++s) {
#pragma unroll
            for (int i = 0; i < kGroups; ++i) {
                if (i == kGroups - 2) stage_barrier();   /* the slot is read; stage s + 1 is there */
                /* after the last full stage: the rest's columns, or stale ones that no link takes */
                read(g[(i + 2) % 4], slot_of(i + 2 < kGroups ? s : s + 1), (i + 2) % kGroups);
                __builtin_amdgcn_sched_barrier(0);
                g[i % 4].links(acc);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else {
        Group<MT> g[2];
        if (full) read(g[0], slot_of(0), 0);
#pragma unroll 1
        for (int s = 0; s < full; ++s) {
#pragma unroll
            for (int i = 0; i < kGroups; ++i) {
                if (i == kGroups - 1) stage_barrier();
                read(g[(i + 1) % 2], slot_of(i + 1 < kGroups ? s : s + 1), (i + 1) % kGroups);
                __builtin_amdgcn_sched_barrier(0);
                g[i % 2].links(acc);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if (rest) {
        const uint8_t *slot = slot_of(full);
        const float *xs = reinterpret_cast<const float *>(slot + kSlotBytes) + wave * MT * kFloatStage;
        for (int c = 0; c < rest; ++c) {
            const float wv = *reinterpret_cast<const float *>(slot + (c >> 2) * kQuadBytes + lane * 16 + 4 * (c & 3));
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = __builtin_fmaf(wv, xs[t * kFloatStage + c], acc[t]);
        }
        stage_barrier();
    }
    const uint32_t row = row0 + lane;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const uint32_t tok = tok0 + wave * MT + t;
        if (row < rows && tok < tokens) y[(size_t)tok * ldy + row] = acc[t];
    }
}

/* One lane per row, its chain element by element: rows that fill the chip by
 * themselves and whose weights cost more to form quad by quad than their links
 * (row_walk says which) */
template <int T, int MT>
__device__ __forceinline__ void float_chain(const uint8_t *row, const float *x, uint32_t width, float *total)
{
    auto step = [&](float wv, uint32_t e) {
#pragma unroll
        for (int t = 0; t < MT; ++t) total[t] = __builtin_fmaf(wv, x[(size_t)t * width + e], total[t]);
    };
    if constexpr (T == kQ8_0) {
        for (uint32_t base = 0; base < width; base += 32, row += 34) {
            const float d = f16_to_f32(ld16(row));
            for (int i = 0; i < 32; ++i) step(fmul_rn(d, (float)(int8_t)row[2 + i]), base + i);
        }
    } else if constexpr (T == kQ2K) {
        for (uint32_t base = 0; base < width; base += 256, row += 84) {
            const float d = f16_to_f32(ld16(row + 80)), dmin = f16_to_f32(ld16(row + 82));
            for (int i = 0; i < 16; ++i) {
                const float scale = fmul_rn(d, (float)(row[i] & 15)), minimum = fmul_rn(dmin, (float)(row[i] >> 4));
                const int half = i / 8, field = (i % 8) / 2, part = i % 2;
                for (int j = 0; j < 16; ++j) {
                    const int q = (row[16 + 32 * half + 16 * part + j] >> (2 * field)) & 3;
                    step(__fsub_rn(fmul_rn(scale, (float)q), minimum), base + 16 * i + j);
                }
            }
        }
    } else {
        constexpr bool five = T == kQ5K;
        for (uint32_t base = 0; base < width; base += 256, row += five ? 176 : 144) {
            const float d = f16_to_f32(ld16(row)), dmin = f16_to_f32(ld16(row + 2));
            const uint8_t *qh = row + 16, *qs = row + (five ? 48 : 16);
            for (int c = 0; c < 4; ++c) {
                int sc0, m0, sc1, m1;
                k4_scale_min(2 * c, row + 4, sc0, m0);
                k4_scale_min(2 * c + 1, row + 4, sc1, m1);
                const float d0 = fmul_rn(d, (float)sc0), mm0 = fmul_rn(dmin, (float)m0);
                const float d1 = fmul_rn(d, (float)sc1), mm1 = fmul_rn(dmin, (float)m1);
                for (int i = 0; i < 32; ++i) {
                    const int q = (qs[32 * c + i] & 15) + (five && ((qh[i] >> (2 * c)) & 1) ? 16 : 0);
                    step(__fsub_rn(fmul_rn(d0, (float)q), mm0), base + 64 * c + i);
                }
                for (int i = 0; i < 32; ++i) {
                    const int q = (qs[32 * c + i] >> 4) + (five && ((qh[i] >> (2 * c + 1)) & 1) ? 16 : 0);
                    step(__fsub_rn(fmul_rn(d1, (float)q), mm1), base + 64 * c + 32 + i);
                }
            }
        }
    }
}

template <int T, int MT>
__global__ __launch_bounds__(256) void gemv_float_rows(const uint8_t *__restrict__ w, const float *__restrict__ x,
                                                       float *__restrict__ y, uint32_t ldy, uint32_t rows,
                                                       uint32_t width, uint64_t row_bytes)
{
    const uint32_t row = blockIdx.x * 256u + threadIdx.x;
    float total[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) total[t] = 0.0f;
    float_chain<T, MT>(w + (size_t)(row < rows ? row : rows - 1) * row_bytes, x, width, total);
#pragma unroll
    for (int t = 0; t < MT; ++t)
        if (row < rows) y[(size_t)t * ldy + row] = total[t];
}

template <int T, int MT, int CW, int ST = 64>
bool launch_float(const uint8_t *w, const float *x, float *y, uint32_t ldy, uint32_t rows, uint32_t width,
                  uint32_t row_bytes, uint32_t tokens, hipStream_t stream)
{
    return launch_kernel(gemm_float_kernel<T, MT, CW, ST>,
                         dim3((rows + kFloatRows - 1) / kFloatRows, (tokens + MT * CW - 1) / (MT * CW)),
                         dim3(64 * CW + kProducers), stream, w, x, y, ldy, rows, width, row_bytes, tokens,
                         stages_of(width, ST));
}

/* Up to eight tokens.  The types of real float matrices (GGUF files keep
 * norms, small projections and Q8_0 models in them) have a kernel per token
 * count, and stages of 128 columns where the matrix gives a compute unit at
 * most one workgroup: half the barriers for the chain that the time is
 * (F16 5120 x 17408, one token: 91 against 127 us), where more rows want the
 * workgroups of smaller stages side by side (F16 34816 x 5120: 78 against
 * 91 us). */
template <int T, int MT>
bool launch_float_few(const uint8_t *w, const float *x, float *y, uint32_t ldy, uint32_t rows, uint32_t width,
                      uint32_t row_bytes, uint32_t tokens, hipStream_t stream)
{
    if constexpr (T == kF32 || T == kF16 || T == kBF16 || T == kQ8_0 || MT <= 3) {
        if ((rows + kFloatRows - 1) / kFloatRows <= 256)
            return launch_float<T, MT, 1, 128>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    }
    return launch_float<T, MT, 1>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
}

/* Tall matrices whose rows one lane each walks: the formats and token counts
 * (kRowTokens at most) whose element loop is the cheaper one, from 65536 rows
 * (a wavefront per SIMD) on.  Workgroups with producers / a lane per row:
 * Q4_K, two tokens, 65536 x 256 and 131072 x 5120 10.3 / 6.2 and 280 / 161 us,
 * one token 131072 x 5120 278 / 246, 248320 x 1024 107 / 120; Q5_K, one token,
 * 65536 x 5120 209 / 189, 248320 x 1024 146 / 110; 65536 x 256, one token, Q2_K
 * 8.5 / 6.8 and Q8_0 10.2 / 8.2; 65536 x 512, two tokens, Q8_0 19 / 17.  At
 * 49152 rows they are even or the producers win (Q4_K 49152 x 512 11.5 / 13.9).
 * Rows of fewer than 256 columns stay with the producers, which lose there on
 * such matrices (Q8_0 248320 x 32, four tokens 14.9 us against 5.1). */
template <int T>
constexpr uint32_t kRowTokens = T == kQ8_0 || T == kQ2K ? 3 : T == kQ4K ? 2 : T == kQ5K ? 1 : 0;
template <int T>
bool row_walk(uint32_t rows, uint32_t width, uint32_t tokens)
{
    if (tokens > kRowTokens<T> || rows < 65536) return false;
    if (T == kQ5K) return true;
    if (T == kQ4K) return tokens == 2 || width <= 256 || rows < 196608;
    return width <= 256 || (T == kQ8_0 && width <= 512 && tokens > 1);
}

template <int T>
bool launch_float_t(const uint8_t *w, const float *x, float *y, uint32_t ldy, uint32_t rows, uint32_t width,
                    uint32_t row_bytes, uint32_t tokens, hipStream_t stream)
{
    if constexpr (kRowTokens<T> > 0) {
        if (row_walk<T>(rows, width, tokens)) {
            const dim3 grid((rows + 255) / 256), block(256);
            if (tokens == 1) return launch_kernel(gemv_float_rows<T, 1>, grid, block, stream, w, x, y, ldy, rows, width, row_bytes);
            if constexpr (kRowTokens<T> > 1) {
                if (tokens == 2) return launch_kernel(gemv_float_rows<T, 2>, grid, block, stream, w, x, y, ldy, rows, width, row_bytes);
            }
            if constexpr (kRowTokens<T> > 2)
                return launch_kernel(gemv_float_rows<T, 3>, grid, block, stream, w, x, y, ldy, rows, width, row_bytes);
        }
    }
    if (tokens == 1) return launch_float_few<T, 1>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    if (tokens == 2) return launch_float_few<T, 2>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    if (tokens == 3) return launch_float_few<T, 3>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    if (tokens <= 4) return launch_float_few<T, 4>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    if (tokens <= 8) return launch_float_few<T, 8>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    /* one pass over the matrix per 32 or 64 tokens, four chain wavefronts */
    if (tokens <= 32) return launch_float<T, 8, 4>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
    return launch_float<T, 16, 4>(w, x, y, ldy, rows, width, row_bytes, tokens, stream);
}

}  // namespace

namespace {

bool launch_float_rows(int type, uint32_t m, const uint8_t *w, const float *x, float *y, uint32_t ldy, uint32_t rows,
                       uint32_t width, uint32_t row_bytes, hipStream_t stream)
{
    switch (type) {
    case kF32: return launch_float_t<kF32>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kF16: return launch_float_t<kF16>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kBF16: return launch_float_t<kBF16>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kQ8_0: return launch_float_t<kQ8_0>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kIQ4NL: return launch_float_t<kIQ4NL>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kQ2K: return launch_float_t<kQ2K>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kQ3K: return launch_float_t<kQ3K>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kQ4K: return launch_float_t<kQ4K>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kQ5K: return launch_float_t<kQ5K>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    case kQ6K: return launch_float_t<kQ6K>(w, x, y, ldy, rows, width, row_bytes, m, stream);
    default: return false;
    }
}

}  // namespace

bool launch_gemm_float(int type, uint32_t m, const uint8_t *w, const float *x, float *y, uint32_t ldy, uint32_t rows,
                       uint32_t width, hipStream_t stream)
{
    uint32_t e = 0, b = 0;
    if (m < 1 || ldy < rows || !rows || !width || !format_block_shape(type, &e, &b) || width % e) return false;
    const uint64_t row_bytes = (uint64_t)width / e * b;
    /* a workgroup addresses its rows with 32-bit offsets and a launch's grid
     * holds 65535 token tiles: wider rows and longer batches take several
     * launches (with one row per launch the stride is not used) */
    const uint64_t fit = 0xffffffffull / row_bytes;
    const uint32_t row_step = fit >= kFloatRows ? rows : fit ? (uint32_t)fit : 1u, token_step = 65535u * 64;
    for (uint32_t r = 0; r < rows;) {
        const uint32_t nr = rows - r < row_step ? rows - r : row_step;
        for (uint32_t t = 0; t < m;) {
            const uint32_t nt = m - t < token_step ? m - t : token_step;
            if (!launch_float_rows(type, nt, w + (size_t)r * row_bytes, x + (size_t)t * width,
                                   y + (size_t)t * ldy + r, ldy, nr, width, (uint32_t)row_bytes, stream))
                return false;
            t += nt;
        }
        r += nr;
    }
    return true;
}

}  // namespace q38
