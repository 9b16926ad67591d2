/* Prompt-length batches (kWideMinTokens tokens and more) of the formats
 * without a wide kernel of their own, against Q8_K activations, on the gfx950
 * matrix cores: Q2_K, Q3_K, Q4_K (row-major), Q5_K, Q6_K, IQ1_S, IQ2_XXS,
 * IQ2_XS, IQ2_S, IQ3_XXS, IQ3_S, IQ4_XS and IQ4_NL.  Weights are the GGUF's
 * own row-major blocks.
 *
 * Arithmetic: per (row, token) the reference's eight AVX2 lane chains
 * acc[l] = fmaf(d_b, W[b][l], acc[l]) over the super-blocks b in order, then
 * ((a0+a4)+(a2+a6)) + ((a1+a5)+(a3+a7)) plus the format's min or correction
 * chain (qwen38_quant.c:510-1253, 1546-1833).  W[b][l] is an exact integer:
 * the sum over the lane's 32 elements (4 of each 32-element group g) of
 * s[g] * q * a.  The products run as two v_mfma_f32_32x32x16_f16 per lane
 * with the weight operand s * q and the activation operand a:
 *  - |s * q| <= 2048 is exact in fp16 for every format but Q6_K and IQ4_XS.
 *    Those split s = 2^k t + u (k = 1 for IQ4_XS, 1 for Q6_K): 2^k t q is a
 *    multiple of 2 of at most 4096 and u q at most 127, both exact, and the
 *    second operand's products accumulate into the same sums;
 *  - every partial sum is an integer of at most 2^24, exact in fp32.
 * Q6_K: the reference forms sum(s q' a) with q' = q + 32 unsigned and takes
 * 32 (s[2l] S[2l] + s[2l+1] S[2l+1]) off lane l, S being the block's sums of
 * 16 activations.  That is 32 (sum_g s[g] A4[g] - s[2l] S[2l] - s[2l+1]
 * S[2l+1]) more than the signed product, A4[g] the sum of the lane's four
 * activations of group g: one more product per lane, added with one fmaf
 * (both terms are exact, so it rounds as the integer's conversion does).
 * Min and correction sums (m[i] * S[i]) are products over the 16 sums (Q4_K:
 * their int16 pair sums), each split into a multiple of 64 and a rest, both
 * exact in fp16.  Their sums stay below 2^24 for any int16 (16 * 15 * 32768 for
 * Q2_K and IQ1_S, 2 * 63 * 32768 for a Q4_K lane's two sub-blocks) but for
 * Q5_K's 16 * 63 * 32768: there the multiples of 64 and the rests are summed
 * apart, below 2^19 steps of 64 and 2^16.
 * IQ4_NL has one fp32 scale per group, so each group's product is taken by
 * itself (v_mfma_f32_32x32x4_2b_f16: two groups per instruction).
 *
 * Layout.  A workgroup of eight wavefronts covers 64 rows x 32 TT tokens and
 * runs the blocks in order, two phases per block:
 *  1. wavefront l decodes lane l of the 64 rows (one row per GPU lane, the
 *     block's bytes from LDS, so all format bit-work has a uniform l) into
 *     fp16 operands in LDS, and all threads convert the tokens' activations:
 *     each weight is decoded once per 32 TT tokens and each activation once
 *     per 64 rows, where a wavefront converting its own operands would do
 *     both twice;
 *  2. wavefront (lane half lh, row half, token half) multiplies its 32 rows
 *     x 16 TT tokens for the AVX2 lanes 4 lh .. 4 lh + 3 and runs their
 *     chains.  The next block's weight bytes are in flight from phase 1 on
 *     and land in LDS at the end of phase 2; its activations are loaded
 *     during phase 2.
 * LDS operands are planes of 16 bytes per row (token): [l][p][row], p = 0..3
 * the pair of groups 2p, 2p + 1, so the reads of a product are conflict-free.
 *
 * Bound.  Two phases between barriers that do not overlap (one workgroup per
 * compute unit: registers and LDS): IQ4_XS, 301 tokens, 34816 rows, vector
 * units 0.49 busy, matrix cores 0.24.  IQ4_XS, 301 tokens: 34816 x 5120
 * 470 us (228 TFLOP/s), 5120 x 17408 219 us, where launches of 8 tokens on
 * the vector units, each decoding the matrix again, took 19.6 and 10.7 ms.
 * 1024 tokens x 34816 x 5120: Q3_K 934 us (391 TFLOP/s), IQ4_XS 1155 us,
 * Q5_K 1715 us, Q6_K 2093 us.  An occupancy of two workgroups (128 VGPRs)
 * spills and measured 2.2 times slower (Q3_K).
 */
#include "q38_format_decode.h"
#include "q38_kernels.h"

namespace q38 {

namespace {

typedef _Float16 half8p __attribute__((ext_vector_type(8)));
typedef _Float16 half4p __attribute__((ext_vector_type(4)));
typedef _Float16 half2p __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f32v __attribute__((ext_vector_type(32)));

constexpr int kPromptRows = 64, kPromptThreads = 512;

template <int T>
struct Prompt {
    static constexpr bool split = T == kQ6K || T == kIQ4XS;
    static constexpr bool min4 = T == kQ4K;
    static constexpr bool scalar = has_extra<T>();
    static constexpr bool sums = min4 || scalar;
    static constexpr bool offset = T == kQ6K;
    static constexpr bool groups = T == kIQ4NL;
};

/* byte offsets of the LDS areas */
template <int T, int TT>
struct PromptLds {
    using P = Prompt<T>;
    static constexpr int tokens = 32 * TT;
    static constexpr int bb = (int)(T == kQ2K ? 84 : T == kQ3K ? 110 : T == kQ4K ? 144 : T == kQ5K ? 176 : T == kQ6K ? 210
                              : T == kIQ2XXS ? 66 : T == kIQ2XS ? 74 : T == kIQ2S ? 82 : T == kIQ3XXS ? 98
                              : T == kIQ3S ? 110 : T == kIQ4XS ? 136 : T == kIQ4NL ? 144 : 50);
    static constexpr int dwords = (bb + 3) / 4;
    static constexpr int raw_stride = 4 * (dwords | 1);             /* odd: a column of dwords hits every bank */
    static constexpr int wplane = kPromptRows * 16, xplane = tokens * 16 + 64;
    static constexpr int w0 = 0;
    static constexpr int w1 = w0 + 32 * wplane;                     /* the second operand of a split scale */
    static constexpr int x0 = w1 + (P::split ? 32 * wplane : 0);
    static constexpr int cw = x0 + 32 * xplane;                     /* Q6_K offset product: [l][2][row], [l][2][token] */
    static constexpr int cx = cw + (P::offset ? 16 * wplane : 0);
    static constexpr int raw = cx + (P::offset ? 16 * tokens * 16 : 0);
    static constexpr int ms = raw + kPromptRows * raw_stride;       /* [4][row] 4 halves: min multipliers */
    static constexpr int ss = ms + (P::sums ? 4 * kPromptRows * 8 : 0);   /* [2][4][token] 4 halves: sums */
    static constexpr int xs = (ss + (P::sums ? 8 * tokens * 8 : 0) + 15) / 16 * 16;   /* [token] scales */
    static constexpr int dd = xs + tokens * 4;                      /* [row] d, then [row] dmin, or [8][row] d */
    static constexpr int stage = dd + kPromptRows * 4 * (P::groups ? 8 : 2);
    static constexpr int values = 4 + (P::min4 ? 2 : P::scalar ? 1 : 0);
    static constexpr int exchange = 4 * 8 * values * 64 * 4;
    static constexpr int bytes = stage > exchange ? stage : exchange;
};

__device__ __forceinline__ half2p hp(uint32_t v) { return __builtin_bit_cast(half2p, v); }

/* four int8 (one dword) as fp16, element order 0, 1, 2, 3 */
__device__ __forceinline__ void bytes_to_half(uint32_t v, half2p &a, half2p &b)
{
    const half2p bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const uint32_t u = v ^ 0x80808080u;
    a = hp(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias;
    b = hp(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias;
}

__device__ __forceinline__ half8p join(half2p a, half2p b, half2p c, half2p d)
{
    half8p v;
    v[0] = a[0]; v[1] = a[1]; v[2] = b[0]; v[3] = b[1];
    v[4] = c[0]; v[5] = c[1]; v[6] = d[0]; v[7] = d[1];
    return v;
}

__device__ __forceinline__ half2p both(int v)
{
    const _Float16 h = (_Float16)(float)v;
    return (half2p){h, h};
}

template <int T, int TT>
__global__ __launch_bounds__(kPromptThreads, 1) void gemm_prompt(const uint8_t *__restrict__ w,
                                                               const uint8_t *__restrict__ x, float *__restrict__ y,
                                                               uint32_t ldy, uint32_t rows, uint32_t nb,
                                                               uint32_t tokens, const uint32_t *__restrict__ iq1s_grid)
{
    using P = Prompt<T>;
    using L = PromptLds<T, TT>;
    constexpr int kSub = TT / 2;                 /* 32-token products per wavefront */
    constexpr int kTok = L::tokens;
    constexpr int kRawItems = (kPromptRows * L::dwords + kPromptThreads - 1) / kPromptThreads;
    constexpr int kActItems = kTok * 8 / kPromptThreads;
    __shared__ __attribute__((aligned(16))) uint8_t lds[L::bytes];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lh = wv & 1, rt = (wv >> 1) & 1, tg = wv >> 2;
    const int r = lane & 31, q = lane >> 5;
    const uint32_t row0 = blockIdx.x * kPromptRows, tok0 = blockIdx.y * kTok;

    /* weight bytes of one block of the 64 rows, dword i of a row's block per
     * item (the last one of a block of 4 k + 2 bytes is two bytes); rows past
     * the matrix repeat the last row */
    const uint8_t *wbase = w + (size_t)row0 * nb * L::bb;
    uint32_t raw_at[kRawItems];
#pragma unroll
    for (int k = 0; k < kRawItems; ++k) {
        const int i = tid + k * kPromptThreads;
        const uint32_t rr = (uint32_t)i / L::dwords < (uint32_t)kPromptRows ? (uint32_t)i / L::dwords : kPromptRows - 1;
        const uint32_t have = rows - row0 - 1;
        raw_at[k] = (rr < have ? rr : have) * nb * L::bb + 4 * ((uint32_t)i % L::dwords);
    }
    auto load_raw = [&](uint32_t b, uint32_t (&v)[kRawItems]) {
        const uint8_t *base = wbase + (size_t)b * L::bb;
#pragma unroll
        for (int k = 0; k < kRawItems; ++k) {
            const int i = tid + k * kPromptThreads;
            v[k] = 0;
            if (i < kPromptRows * L::dwords) {
                const uint8_t *p = base + raw_at[k];
                if (L::bb % 4 == 0 || i % L::dwords != L::dwords - 1) __builtin_memcpy(&v[k], p, 4);
                else v[k] = ld16(p);
            }
        }
    };
    auto store_raw = [&](const uint32_t (&v)[kRawItems]) {
#pragma unroll
        for (int k = 0; k < kRawItems; ++k) {
            const int i = tid + k * kPromptThreads;
            if (i < kPromptRows * L::dwords)
                *reinterpret_cast<uint32_t *>(lds + L::raw + (i / L::dwords) * L::raw_stride + 4 * (i % L::dwords)) = v[k];
        }
    };

    /* activations: item = (token, group), eight lanes per token; tokens past
     * the batch repeat the last one */
    struct Act {
        uint32_t v[kActItems][8];
        float scale;        /* of token tid, tid < kTok */
        uint32_t sums[4];   /* sums 8 (tid / kTok) .. of token tid % kTok, tid < 2 kTok */
    };
    auto token_block = [&](int t, uint32_t b) {
        const uint32_t tok = tok0 + t < tokens ? tok0 + t : tokens - 1;
        return x + ((size_t)tok * nb + b) * kQ8KBytes;
    };
    auto load_act = [&](uint32_t b, Act &a) {
#pragma unroll
        for (int k = 0; k < kActItems; ++k) {
            const int i = tid + k * kPromptThreads;
            const uint32_t *p = reinterpret_cast<const uint32_t *>(token_block(i >> 3, b) + 4 + 32 * (i & 7));
#pragma unroll
            for (int e = 0; e < 8; ++e) a.v[k][e] = p[e];
        }
        if (tid < kTok) a.scale = *reinterpret_cast<const float *>(token_block(tid, b));
        if (P::sums || P::offset) {
            if (tid < 2 * kTok) {
                const uint32_t *p = reinterpret_cast<const uint32_t *>(token_block(tid % kTok, b) + 260 + 16 * (tid / kTok));
#pragma unroll
                for (int e = 0; e < 4; ++e) a.sums[e] = p[e];
            }
        }
    };
    auto store_act = [&](const Act &a) {
#pragma unroll
        for (int k = 0; k < kActItems; ++k) {
            const int i = tid + k * kPromptThreads, t = i >> 3, g = i & 7;
            uint8_t *base = lds + L::x0 + (g >> 1) * L::xplane + t * 16 + (g & 1) * 8;
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                half2p u, v;
                bytes_to_half(a.v[k][l], u, v);
                *reinterpret_cast<uint2 *>(base + 4 * l * L::xplane) =
                    make_uint2(__builtin_bit_cast(uint32_t, u), __builtin_bit_cast(uint32_t, v));
                if constexpr (P::offset) {
                    const int sum4 = dot4z((int)a.v[k][l], 0x01010101);
                    *reinterpret_cast<_Float16 *>(lds + L::cx + (2 * l * kTok + t) * 16 + 2 * g) = (_Float16)(float)sum4;
                }
            }
        }
        if (tid < kTok) *reinterpret_cast<float *>(lds + L::xs + 4 * tid) = a.scale;
        if (tid < 2 * kTok) {
            const int t = tid % kTok, hi = tid / kTok;
            if constexpr (P::sums) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    half4p high = {}, rest = {};
                    if constexpr (P::min4) {
                        /* the reference adds pairs of sums in int16 */
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            const uint32_t v = a.sums[2 * i + e];
                            const int s = (int16_t)((v & 0xffffu) + (v >> 16));
                            const _Float16 hi64 = (_Float16)(float)(s & ~63), low64 = (_Float16)(float)(s & 63);
                            (e ? rest : high)[2 * e] = hi64;
                            (e ? rest : high)[2 * e + 1] = low64;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int s = (int16_t)(a.sums[2 * i + (e >> 1)] >> (16 * (e & 1)));
                            high[e] = (_Float16)(float)(s & ~63);
                            rest[e] = (_Float16)(float)(s & 63);
                        }
                    }
                    *reinterpret_cast<half4p *>(lds + L::ss + ((2 * hi + i) * kTok + t) * 8) = high;
                    *reinterpret_cast<half4p *>(lds + L::ss + ((4 + 2 * hi + i) * kTok + t) * 8) = rest;
                }
            }
            if constexpr (P::offset) {
                /* lane l subtracts s[2l] S[2l] + s[2l+1] S[2l+1]: S as a
                 * multiple of 64 and a rest */
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    half8p v = {};
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int s = (int16_t)(a.sums[i] >> (16 * e));
                        v[e] = (_Float16)(float)-(s & ~63);
                        v[2 + e] = (_Float16)(float)-(s & 63);
                    }
                    *reinterpret_cast<half8p *>(lds + L::cx + ((2 * (4 * hi + i) + 1) * kTok + t) * 16) = v;
                }
            }
        }
    };

    /* phase 1: lane l = wv of row `lane` */
    auto decode = [&]() {
        const uint8_t *blk = lds + L::raw + lane * L::raw_stride;
        LaneBlock lb;
        decode_lane<T>(blk, wv, table_of<T>(iq1s_grid), lb);
        uint8_t *out = lds + L::w0 + 4 * wv * L::wplane + lane * 16;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            half2p a[4];
            bytes_to_half(lb.q[2 * p], a[0], a[1]);
            bytes_to_half(lb.q[2 * p + 1], a[2], a[3]);
            const int s0 = lb.s[2 * p], s1 = lb.s[2 * p + 1];
            if constexpr (P::split) {
                const half2p h0 = both(s0 & ~1), h1 = both(s1 & ~1), u0 = both(s0 & 1), u1 = both(s1 & 1);
                *reinterpret_cast<half8p *>(out + p * L::wplane) = join(a[0] * h0, a[1] * h0, a[2] * h1, a[3] * h1);
                *reinterpret_cast<half8p *>(out + (L::w1 - L::w0) + p * L::wplane) =
                    join(a[0] * u0, a[1] * u0, a[2] * u1, a[3] * u1);
            } else if constexpr (P::groups) {
                *reinterpret_cast<half8p *>(out + p * L::wplane) = join(a[0], a[1], a[2], a[3]);
            } else {
                const half2p h0 = both(s0), h1 = both(s1);
                *reinterpret_cast<half8p *>(out + p * L::wplane) = join(a[0] * h0, a[1] * h0, a[2] * h1, a[3] * h1);
            }
        }
        float *d = reinterpret_cast<float *>(lds + L::dd) + lane;
        if constexpr (P::groups) {
            d[kPromptRows * wv] = f16_to_f32(ld16(blk + 18 * wv));
        } else {
            if (wv == 0) d[0] = lb.d;
            if constexpr (P::min4 || T == kQ2K || T == kQ5K) {
                if (wv == 1) d[kPromptRows] = lb.dmin;
            }
        }
        if constexpr (P::offset) {
            half8p c;
#pragma unroll
            for (int g = 0; g < 8; ++g) c[g] = (_Float16)(float)lb.s[g];
            *reinterpret_cast<half8p *>(lds + L::cw + (2 * wv * kPromptRows + lane) * 16) = c;
            const int s0 = (int8_t)blk[192 + 2 * wv], s1 = (int8_t)blk[193 + 2 * wv];
            half8p e = {};
            e[0] = e[2] = (_Float16)(float)s0;
            e[1] = e[3] = (_Float16)(float)s1;
            *reinterpret_cast<half8p *>(lds + L::cw + ((2 * wv + 1) * kPromptRows + lane) * 16) = e;
        }
        if constexpr (P::sums) {
            if (wv >= 4) {
                const int i = wv - 4;   /* the multipliers of sums 4i .. 4i + 3 */
                half4p m;
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    int m0, m1;
                    extra_factors<T>(blk, 2 * i + e, m0, m1);
                    m[2 * e] = (_Float16)(float)m0;
                    m[2 * e + 1] = (_Float16)(float)m1;
                }
                *reinterpret_cast<half4p *>(lds + L::ms + (i * kPromptRows + lane) * 8) = m;
            }
        }
    };

    /* chains: the four AVX2 lanes of the wavefront's half, and the min lanes
     * 2 lh, 2 lh + 1 (min4), or the scalar min / correction chain, which lane
     * half lh runs for one product: with two products each half takes one */
    float acc[kSub][4][16], extra[P::min4 ? 2 : 1][16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int u = 0; u < kSub; ++u) acc[u][k][j] = 0.0f;
        extra[0][j] = 0.0f;
        if constexpr (P::min4) extra[1][j] = 0.0f;
    }

    uint32_t raw[kRawItems];
    Act act;
    load_raw(0, raw);
    load_act(0, act);
    store_raw(raw);
    __syncthreads();
    const int wrow = 32 * rt + r;
#pragma unroll 1
    for (uint32_t b = 0; b < nb; ++b) {
        const uint32_t next = b + 1 < nb ? b + 1 : b;
        load_raw(next, raw);
        decode();
        store_act(act);
        __syncthreads();
        load_act(next, act);
        const float *dl = reinterpret_cast<const float *>(lds + L::dd) + wrow;
        const uint8_t *wl = lds + L::w0 + (16 * lh + q) * L::wplane + wrow * 16;
#pragma unroll
        for (int u = 0; u < kSub; ++u) {
            const int tt = tg * kSub + u;   /* 32-token tile of the workgroup */
            const uint8_t *xl = lds + L::x0 + (16 * lh + q) * L::xplane + (32 * tt + r) * 16;
            float xsv[16];
#pragma unroll
            for (int j = 0; j < 16; ++j)
                xsv[j] = reinterpret_cast<const float *>(lds + L::xs)[32 * tt + 8 * (j >> 2) + 4 * q + (j & 3)];
            if constexpr (P::groups) {
                /* lane half q holds group 2p + q of the product: the first
                 * sixteen results are group 2p's, the others 2p + 1's */
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    float d0[16], d1[16];
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        d0[j] = fmul_rn(dl[kPromptRows * 2 * p], xsv[j]);
                        d1[j] = fmul_rn(dl[kPromptRows * (2 * p + 1)], xsv[j]);
                    }
                    const uint8_t *wp = lds + L::w0 + (16 * lh + p) * L::wplane + wrow * 16 + 8 * q;
                    const uint8_t *xp = lds + L::x0 + (16 * lh + p) * L::xplane + (32 * tt + r) * 16 + 8 * q;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const half4p bw = *reinterpret_cast<const half4p *>(wp + 4 * k * L::wplane);
                        const half4p ax = *reinterpret_cast<const half4p *>(xp + 4 * k * L::xplane);
                        const f32v z = {};
                        const f32v g = __builtin_amdgcn_mfma_f32_32x32x4f16(ax, bw, z, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 16; ++j) {
                            acc[u][k][j] = __builtin_fmaf(d0[j], g[j], acc[u][k][j]);
                            acc[u][k][j] = __builtin_fmaf(d1[j], g[16 + j], acc[u][k][j]);
                            asm volatile("" : "+v"(acc[u][k][j]));
                        }
                    }
                }
            } else {
                float dx[16];
#pragma unroll
                for (int j = 0; j < 16; ++j) dx[j] = fmul_rn(dl[0], xsv[j]);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const half8p a0 = *reinterpret_cast<const half8p *>(xl + 4 * k * L::xplane);
                    const half8p a1 = *reinterpret_cast<const half8p *>(xl + (4 * k + 2) * L::xplane);
                    const half8p b0 = *reinterpret_cast<const half8p *>(wl + 4 * k * L::wplane);
                    const half8p b1 = *reinterpret_cast<const half8p *>(wl + (4 * k + 2) * L::wplane);
                    const f16v z = {};
                    f16v g = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, b0, z, 0, 0, 0);
                    g = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b1, g, 0, 0, 0);
                    if constexpr (P::split) {
                        const half8p c0 = *reinterpret_cast<const half8p *>(wl + L::w1 + 4 * k * L::wplane);
                        const half8p c1 = *reinterpret_cast<const half8p *>(wl + L::w1 + (4 * k + 2) * L::wplane);
                        g = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, c0, g, 0, 0, 0);
                        g = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, c1, g, 0, 0, 0);
                    }
                    if constexpr (P::offset) {
                        const int l = 4 * lh + k;
                        const half8p ca = *reinterpret_cast<const half8p *>(lds + L::cx + ((2 * l + q) * kTok + 32 * tt + r) * 16);
                        const half8p cb = *reinterpret_cast<const half8p *>(lds + L::cw + ((2 * l + q) * kPromptRows + wrow) * 16);
                        const f16v c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ca, cb, z, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 16; ++j) g[j] = __builtin_fmaf(32.0f, c[j], g[j]);
                    }
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        acc[u][k][j] = __builtin_fmaf(dx[j], g[j], acc[u][k][j]);
                        /* the link stays here: the compiler would sink it
                         * past the barrier and keep the products instead */
                        asm volatile("" : "+v"(acc[u][k][j]));
                    }
                }
                if constexpr (P::min4) {
                    /* min lanes 2 lh, 2 lh + 1: the first pair of sums in lane
                     * half 0, the second in lane half 1 */
                    float dm[16];
#pragma unroll
                    for (int j = 0; j < 16; ++j) dm[j] = -fmul_rn(dl[kPromptRows], xsv[j]);
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const int i = 2 * lh + k;
                        const half4p sa = *reinterpret_cast<const half4p *>(lds + L::ss + ((4 * q + i) * kTok + 32 * tt + r) * 8);
                        const half4p sb = *reinterpret_cast<const half4p *>(lds + L::ms + (i * kPromptRows + wrow) * 8);
                        const f16v z = {};
                        const f16v m = __builtin_amdgcn_mfma_f32_32x32x8f16(sa, sb, z, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 16; ++j) {
                            extra[k][j] = __builtin_fmaf(dm[j], m[j], extra[k][j]);
                            asm volatile("" : "+v"(extra[k][j]));
                        }
                    }
                }
                if constexpr (P::scalar) {
                    if (lh == (kSub == 2 ? u : 1)) {
                        auto sums4 = [&](int k) {
                            return *reinterpret_cast<const half4p *>(lds + L::ss + (k * kTok + 32 * tt + r) * 8);
                        };
                        auto factors4 = [&](int k) {
                            return *reinterpret_cast<const half4p *>(lds + L::ms + (k * kPromptRows + wrow) * 8);
                        };
                        f16v m = {};
                        if constexpr (T == kQ5K) {
                            f16v low = {};
#pragma unroll
                            for (int i = 0; i < 2; ++i) {
                                m = __builtin_amdgcn_mfma_f32_32x32x8f16(sums4(2 * i + q), factors4(2 * i + q), m, 0, 0, 0);
                                low = __builtin_amdgcn_mfma_f32_32x32x8f16(sums4(4 + 2 * i + q), factors4(2 * i + q), low, 0, 0, 0);
                            }
                            /* both exact: one rounding, as the integer sum's conversion */
#pragma unroll
                            for (int j = 0; j < 16; ++j) m[j] = fadd_rn(m[j], low[j]);
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                m = __builtin_amdgcn_mfma_f32_32x32x8f16(sums4(4 * q + i), factors4(i), m, 0, 0, 0);
                        }
#pragma unroll
                        for (int j = 0; j < 16; ++j) {
                            if constexpr (T == kIQ1S) extra[0][j] = fadd_rn(extra[0][j], fmul_rn(dx[j], m[j]));
                            else extra[0][j] = __builtin_fmaf(-fmul_rn(dl[kPromptRows], xsv[j]), m[j], extra[0][j]);
                            asm volatile("" : "+v"(extra[0][j]));
                        }
                    }
                }
            }
        }
        store_raw(raw);
        __syncthreads();
    }

    /* final tree: lane half lh = 1 hands its values over through LDS, eight
     * tokens of a 32-token tile at a time */
    float *xch = reinterpret_cast<float *>(lds) + (size_t)(wv >> 1) * 8 * L::values * 64 + lane;
    const uint32_t row = row0 + wrow;
#pragma unroll
    for (int u = 0; u < kSub; ++u) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            __syncthreads();
            if (lh) {
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    const int j = 8 * half + jj;
                    float *e = xch + jj * L::values * 64;
#pragma unroll
                    for (int k = 0; k < 4; ++k) e[64 * k] = acc[u][k][j];
                    if constexpr (P::sums) e[256] = extra[0][j];
                    if constexpr (P::min4) e[320] = extra[1][j];
                }
            }
            __syncthreads();
            if (!lh) {
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    const int j = 8 * half + jj;
                    const float *e = xch + jj * L::values * 64;
                    float s = fadd_rn(fadd_rn(fadd_rn(acc[u][0][j], e[0]), fadd_rn(acc[u][2][j], e[128])),
                                      fadd_rn(fadd_rn(acc[u][1][j], e[64]), fadd_rn(acc[u][3][j], e[192])));
                    if constexpr (P::min4)
                        s = fadd_rn(s, fadd_rn(fadd_rn(extra[0][j], e[256]), fadd_rn(extra[1][j], e[320])));
                    else if constexpr (P::scalar) {
                        const float c = kSub == 2 && u == 0 ? extra[0][j] : e[256];
                        s = fadd_rn(s, T == kIQ1S ? fmul_rn(0.125f, c) : c);
                    }
                    const uint32_t tok = tok0 + 32 * (tg * kSub + u) + 8 * (j >> 2) + 4 * q + (j & 3);
                    if (row < rows && tok < tokens) y[(size_t)tok * ldy + row] = s;
                }
            }
        }
    }
}

template <int T, int TT>
bool launch_prompt(const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows, uint32_t nb,
                   uint32_t tokens, const void *grid, hipStream_t stream)
{
    static_assert(PromptLds<T, TT>::bytes <= 160 * 1024, "LDS");
    return launch_kernel(gemm_prompt<T, TT>,
                         dim3((rows + kPromptRows - 1) / kPromptRows, (tokens + 32 * TT - 1) / (32 * TT)),
                         dim3(kPromptThreads), stream, w, x, y, ldy, rows, nb, tokens,
                         static_cast<const uint32_t *>(grid));
}

/* Workgroups of 128 tokens where their registers hold (no min lanes, offset
 * product or group chains; Q2_K and Q5_K spill: Q5_K, 34816 x 5120, 301
 * tokens 702 against 558 us) and the batch fills the chip with them: one takes
 * about 1.5 times a 64-token workgroup's time (IQ4_XS, 17408 columns: 217
 * against 152 us for one round of workgroups), so they pay when they need at
 * most two thirds of the rounds over the 256 compute units.  IQ4_XS, 34816 x
 * 5120: 301 tokens 470 against 509 us, 1024 tokens 1155 against 1567 us; on
 * 5120 x 17408 128 tokens 217 against 152 us, so one round stays at 64. */
template <int T>
bool launch_prompt_t(const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows, uint32_t nb,
                     uint32_t tokens, const void *grid, hipStream_t stream)
{
    if constexpr (!Prompt<T>::min4 && !Prompt<T>::offset && !Prompt<T>::groups && T != kQ5K && T != kQ2K) {
        const uint64_t tiles = (rows + kPromptRows - 1) / kPromptRows;
        const uint64_t rounds64 = (tiles * ((tokens + 63) / 64) + 255) / 256;
        const uint64_t rounds128 = (tiles * ((tokens + 127) / 128) + 255) / 256;
        if (3 * rounds128 <= 2 * rounds64) return launch_prompt<T, 4>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    }
    return launch_prompt<T, 2>(w, x, y, ldy, rows, nb, tokens, grid, stream);
}

}  // namespace

/* The most tokens of a batch that launches of up to eight take in less time
 * than one launch here.  A round of these workgroups takes 1.8 (Q4_K) to 2.9 us
 * (Q6_K) per block column whatever the token count, so it loses on
 *  - Q4_K and Q6_K matrices too small to fill the chip (launches / prompt:
 *    1024 x 5120, 9 and 17 tokens 22 / 43 and 38 / 43 us Q4_K, 25 / 61 and 43 /
 *    61 Q6_K; 24 tokens 82 / 39 Q4_K on 2048 rows, but 49 / 61 Q6_K on 512 and
 *    54 / 61 on 1024; 25 tokens 55 / 61 on 512; 4096 x 5120 Q6_K 9 and 12 tokens
 *    54 / 62 and 65 / 62; one row of 17408, 24 and 40 tokens 113 / 198 and 189 /
 *    198 Q6_K, 25 tokens 107 / 120 Q4_K), while 34816 x 5120 at nine tokens
 *    takes 370 / 128 and 337 / 184 us;
 *  - short rows of tall matrices of the other formats, where the few-token
 *    kernel walks a row with eight lanes (248320 x 256, 9 and 16 tokens IQ4_NL
 *    48 / 112 and 69 / 115 us; 34816 x 512, 9 tokens 17 / 33).
 * The other formats' launches are not slower than a round at 9 to about 16
 * tokens of up to 16384 rows either (5120 x 17408, eight tokens of Q5_K 58 us
 * against 155 for a round), which this rule leaves to the round. */
static uint32_t few_token_limit(int type, uint32_t rows, uint32_t nb)
{
    if (type == kQ4K) return rows == 1 && nb > 40 ? 25 : rows < 4096 ? 23 : 8;
    if (type == kQ6K) {
        if (rows == 1 && nb > 40) return 40;
        if (rows <= 1024 && nb >= 8) return nb < 20 ? 24 : rows <= 512 ? 26 : 25;
        return rows < 4096 ? 23 : rows < 4800 ? 10 : 8;
    }
    return rows > 16384 && nb <= 2 ? (nb == 1 ? 16 : 12) : 8;
}

bool prompt_takes(int type, uint32_t tokens, uint32_t rows, uint32_t nb)
{
    if (!format_takes_q8k(type) || type == kIQ1M || !rows || !nb || tokens < (uint32_t)kWideMinTokens) return false;
    /* 32-bit byte offsets inside a workgroup's rows, and the grid's limits */
    if (nb > 65536 || tokens > 65535u * 64) return false;
    return tokens > few_token_limit(type, rows, nb);
}

bool launch_gemm_prompt(int type, uint32_t tokens, const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy,
                        uint32_t rows, uint32_t nb, const void *grid, hipStream_t stream)
{
    if (ldy < rows || !prompt_takes(type, tokens, rows, nb)) return false;
    switch (type) {
    case kQ2K: return launch_prompt_t<kQ2K>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kQ3K: return launch_prompt_t<kQ3K>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kQ4K: return launch_prompt_t<kQ4K>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kQ5K: return launch_prompt_t<kQ5K>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kQ6K: return launch_prompt_t<kQ6K>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ2XXS: return launch_prompt_t<kIQ2XXS>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ2XS: return launch_prompt_t<kIQ2XS>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ2S: return launch_prompt_t<kIQ2S>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ3XXS: return launch_prompt_t<kIQ3XXS>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ3S: return launch_prompt_t<kIQ3S>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ4XS: return launch_prompt_t<kIQ4XS>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ4NL: return launch_prompt_t<kIQ4NL>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    case kIQ1S: return grid && launch_prompt_t<kIQ1S>(w, x, y, ldy, rows, nb, tokens, grid, stream);
    default: return false;
    }
}

}  // namespace q38
