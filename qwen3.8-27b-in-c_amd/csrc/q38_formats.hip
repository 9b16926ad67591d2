/* GEMV / small-M GEMM and row decode for the remaining
 * GGUF matrix formats of the reference model (src/qwen38/qwen38_model.c:
 * 172-189): Q2_K, Q3_K, Q5_K, IQ2_XXS, IQ2_XS, IQ2_S, IQ3_XXS, IQ3_S,
 * IQ4_XS, IQ4_NL, IQ1_S against Q8_K activations.
 *
 * Q8_K path.  Each of the reference's AVX2 kernels (qwen38_quant.c:510-1253,
 * 1636-1725) keeps eight fp32 lanes per row; for every super-block, lane l
 * gets d * W[l], where W[l] is the exact integer sum over bytes 4l..4l+3 of
 * each 32-element group, each group-half scaled by its integer sub-block
 * scale.  Here eight GPU lanes stand for a row's eight accumulators (a
 * wavefront holds eight rows): each decodes the four weights of each group
 * it needs into a packed int8 dword (grid value and sign folded in),
 * multiplies with v_dot4_i32_i8 against the activation dword, scales, and a
 * wavefront runs the fmaf chains.  The eight lanes then add in the reference's tree
 * ((a0 + a4) + (a2 + a6)) + ((a1 + a5) + (a3 + a7)); Q2_K and Q5_K add their
 * scalar min chain, IQ1_S 0.125 times its scalar correction sum, and IQ4_NL
 * applies one fp32 scale per 32-element group (eight FMAs per block).
 *
 * Row decode (q38_tensor_row_f32, :3185-3223): F32 copied, F16 / BF16
 * converted; otherwise each element is the float dot of its block with a
 * unit vector, which is the element's weight expression (a -0 result
 * becoming +0 through the +0 accumulator), or NaN when another weight of
 * the block is not finite (its product with 0 is NaN; written with the bit
 * pattern x86 gives, 0xffc00000).
 */
#include "q38_device.h"
#include "q38_format_decode.h"
#include "q38_kernels.h"

namespace q38 {

namespace {

/* Q8_K path for up to eight tokens: y[t * ldy + row].
 *
 * A workgroup covers eight rows; its H wavefronts split the blocks,
 * lane (row r of eight, AVX2 lane l) of each forming the exact integer sums
 * of its blocks for every token.  The sums (as fp32, exact) and the blocks'
 * scales go through LDS, and wavefront t runs token t's fp32 chains over the
 * blocks in order: the integer work of a row is spread over H wavefronts, so
 * that enough loads are in flight on matrices of few rows, and the order of
 * the fp32 work stays.  Long rows take several phases of at most kBlocks
 * blocks.  The IQ codebooks are copied to LDS: a lookup per four weights is
 * most of these formats' work, and from global memory each costs a cache
 * access per lane.
 *
 * Bound.  Latency of the decode and of the lanes' activation loads (Q5_K, one
 * token, 34816 x 5120: vector units 0.59 busy, wavefronts waiting 0.57 of their
 * time, half of that for issue).  One token,
 * 34816 x 5120 / 5120 x 17408: Q5_K 28 / 19 us (4.4 / 3.1 TB/s), Q3_K 31 / 20,
 * IQ3_S 43 / 29, IQ2_S 54 / 34, IQ1_S 40 / 27 us; eight lanes per row walking
 * all its blocks took 31 / 51, 32 / 49, 77 / 70, 80 / 72 and 77 / 75 us.
 * Eight tokens: Q5_K 89 / 58 us (248 / 622 before), IQ3_S 85 / 57 (237 / 499).
 * H = 8 up to three tokens and 12 for more or for three tokens of long rows:
 * of 4, 8, 12 and 16 wavefronts Q5_K takes 20 / 19 / 19 / 19 us (one token,
 * 17408 columns), 84 / 44 / 51 / 76 us (three tokens, 34816 rows), Q3_K 38
 * (8) and 30 us (12) for three tokens of 17408 columns; 16 or 32 rows per
 * workgroup measured slower on 5120 rows (25 to 48 us for Q3_K). */
template <int T, int MT>
struct GemvFormat {
    static constexpr int table = table_dwords<T>() * 4;
    static constexpr int scalars = T == kIQ1S ? 2 : has_extra<T>() ? 3 : 1;   /* floats per row and block */
    static constexpr int per_block = MT * (64 + scalars * 8) * 4;
    static constexpr int kBlocks = (64 * 1024 - table) / per_block;           /* blocks of a phase at most */
};

/* the block's integer min or correction sum of the lane's row: two products
 * per lane, added over the row's eight lanes */
__device__ __forceinline__ int row_extra(const uint8_t *xb, int l, int m0, int m1)
{
    const int pair = *reinterpret_cast<const int *>(xb + 260 + 4 * l);
    const int sum = quad_sum(m0 * (int)(int16_t)pair + m1 * (pair >> 16));
    return sum + dpp_move<0x141>(0, sum);   /* the row's other quad */
}

template <int T, int MT, int H>
__global__ __launch_bounds__(64 * H) void gemv_format_kernel(const uint8_t *__restrict__ w,
                                                                const uint8_t *__restrict__ x, float *__restrict__ y,
                                                                uint32_t ldy, uint32_t rows, uint32_t nb,
                                                                uint32_t phase_blocks,
                                                                const uint32_t *__restrict__ iq1s_grid)
{
    static_assert(T != kIQ4NL, "IQ4_NL has a scale per group: gemv_rows_kernel");
    using F = GemvFormat<T, MT>;
    constexpr uint32_t kBytes = block_bytes<T>();
    constexpr int kMine = (MT + H - 1) / H;   /* tokens whose chains a wavefront runs */
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   /* table + phase_blocks * per_block bytes */
    uint32_t *table = reinterpret_cast<uint32_t *>(lds);
    /* [block][token][lane], then [block][token][scalar][row] */
    float *sum_s = reinterpret_cast<float *>(lds + F::table);
    float *scalar_s = sum_s + phase_blocks * MT * 64;
    const int lane = threadIdx.x & 63, l = lane & 7, r = lane >> 3;
    const int h = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const uint32_t row = blockIdx.x * 8 + r;
    const uint8_t *wr = w + (size_t)(row < rows ? row : rows - 1) * nb * kBytes;
    if constexpr (F::table > 0) {
        const uint32_t *src = table_of<T>(iq1s_grid);
        for (int i = threadIdx.x; i < table_dwords<T>(); i += 64 * H) table[i] = src[i];
        __syncthreads();
    }
    float acc[kMine], scalar[kMine];
#pragma unroll
    for (int i = 0; i < kMine; ++i) acc[i] = scalar[i] = 0.0f;

    for (uint32_t b0 = 0; b0 < nb; b0 += phase_blocks) {
        const int count = (int)(nb - b0 < phase_blocks ? nb - b0 : phase_blocks);
        const int first = count * h / H, last = count * (h + 1) / H;
#pragma unroll 2
        for (int i = first; i < last; ++i) {
            const uint32_t b = b0 + i;
            const uint8_t *blk = wr + (size_t)b * kBytes;
            LaneBlock lb;
            decode_lane<T>(blk, l, table, lb);
            int m0 = 0, m1 = 0;
            if constexpr (has_extra<T>()) extra_factors<T>(blk, l, m0, m1);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const uint8_t *xb = x + ((size_t)t * nb + b) * kQ8KBytes;
                const float xs = *reinterpret_cast<const float *>(xb);
                const int *aq = reinterpret_cast<const int *>(xb + 4) + l;
                float *so = sum_s + (size_t)(i * MT + t) * 64 + lane;
                float *co = scalar_s + (size_t)(i * MT + t) * F::scalars * 8 + r;
                int wsum = 0;
#pragma unroll
                for (int g = 0; g < 8; ++g) wsum = mad24(lb.s[g], dot4z((int)lb.q[g], aq[8 * g]), wsum);
                *so = (float)wsum;
                int extra = 0;
                if constexpr (has_extra<T>()) extra = row_extra(xb, l, m0, m1);
                if (l == 0) {
                    const float d = fmul_rn(lb.d, xs);
                    co[0] = d;
                    if constexpr (T == kIQ1S) {
                        co[8] = fmul_rn(d, (float)extra);
                    } else if constexpr (has_extra<T>()) {
                        co[8] = -fmul_rn(lb.dmin, xs);
                        co[16] = (float)extra;
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kMine; ++k) {
            const int t = h + k * H;
            if (t >= MT) break;
            const float *so = sum_s + (size_t)t * 64 + lane;
            const float *co = scalar_s + (size_t)t * F::scalars * 8 + r;
#pragma unroll 4
            for (int i = 0; i < count; ++i, so += MT * 64, co += MT * F::scalars * 8) {
                acc[k] = __builtin_fmaf(co[0], so[0], acc[k]);
                if constexpr (T == kIQ1S) scalar[k] = fadd_rn(scalar[k], co[8]);
                else if constexpr (has_extra<T>()) scalar[k] = __builtin_fmaf(co[8], co[16], scalar[k]);
            }
        }
        if (b0 + phase_blocks < nb) __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < kMine; ++k) {
        const int t = h + k * H;
        if (t >= MT) break;
        /* ((a0 + a4) + (a2 + a6)) + ((a1 + a5) + (a3 + a7)), qwen38_quant.c:303-310 */
        float v = fadd_rn(acc[k], __shfl_xor(acc[k], 4, 64));
        v = fadd_rn(v, __shfl_xor(v, 2, 64));
        v = fadd_rn(v, __shfl_xor(v, 1, 64));
        if constexpr (T == kIQ1S) v = fadd_rn(v, fmul_rn(0.125f, scalar[k]));
        else if constexpr (has_extra<T>()) v = fadd_rn(v, scalar[k]);
        if (l == 0 && row < rows) y[(size_t)t * ldy + row] = v;
    }
}

/* decode_lane for gemv_rows_kernel: with few blocks to a row, formats with
 * several header fields per group are faster loading the bytes a lane uses than
 * whole headers to shift them from (65536 x 1024, one token: IQ2_S 27 against
 * 32 us, IQ1_S 26 against 28 us).  m (IQ1_S): the factor of activation sums 2l
 * and 2l + 1, from the header of group l that the lane has anyway. */
template <int T>
__device__ __forceinline__ void decode_walk(const uint8_t *blk, int l, const uint32_t *table, LaneBlock &b, int &m)
{
    const int sec = l >> 1, half = l & 1;
    if constexpr (T == kIQ2S) {
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t index = blk[2 + 4 * g + sec] | (((uint32_t)blk[66 + g] << (8 - 2 * sec)) & 0x300u);
            b.q[g] = negate_bytes(table[2 * index + half], byte_mask4((uint32_t)blk[34 + 4 * g + sec] >> (4 * half)));
            b.s[g] = 1 + 2 * (int)(((uint32_t)blk[74 + g] >> (l & 4)) & 15u);
        }
        b.d = 0.125f * f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ3S) {
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t index = blk[2 + 8 * g + l] | (((uint32_t)(blk[66 + g] >> l) & 1u) << 8);
            b.q[g] = negate_bytes(table[index], byte_mask4((uint32_t)blk[74 + 4 * g + sec] >> (4 * half)));
            b.s[g] = 1 + 2 * (int)((blk[106 + g / 2] >> (4 * (g & 1))) & 15u);
        }
        b.d = f16_to_f32(ld16(blk));
    } else if constexpr (T == kIQ1S) {
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t high = ld16(blk + 34 + 2 * g);
            const uint32_t index = blk[2 + 4 * g + sec] | (((high >> (3 * sec)) & 7u) << 8);
            b.q[g] = table[2 * index + half];
            b.s[g] = 1 + 2 * (int)((high >> 12) & 7u);
            if (l == g) m = high & 0x8000u ? -b.s[g] : b.s[g];
        }
        b.d = f16_to_f32(ld16(blk));
    } else if constexpr (T == kQ3K) {
        const int hi = l >= 4;
        const uint32_t hm = ld32u(blk + 4 * l);
        const uint32_t d0 = ld32u(blk + 32 + 4 * l), d1 = ld32u(blk + 64 + 4 * l);
        const uint8_t *sc = blk + 96;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const uint32_t low = ((g < 4 ? d0 : d1) >> (2 * (g & 3))) & 0x03030303u;
            const uint32_t absent = ~(hm >> g) & 0x01010101u;
            b.q[g] = low + absent * 0xfcu;
            const int i = 2 * g + hi;
            const int lo4 = g < 4 ? sc[i] & 15 : sc[i - 8] >> 4;
            const int hi2 = (sc[8 + i % 4] >> (2 * (i / 4))) & 3;
            b.s[g] = (lo4 | hi2 << 4) - 32;
        }
        b.d = f16_to_f32(ld16(blk + 108));
    } else {
        decode_lane<T>(blk, l, table, b);
    }
}

/* The same for short rows of tall matrices, and for IQ4_NL at any length:
 * eight lanes per row, each running its chain over all blocks, 32 rows per
 * workgroup, the codebooks read from global memory.  Where rows fill the chip
 * by themselves, a workgroup per eight of them costs more than it spreads: its
 * wavefronts have a block each or none, and every one copies the codebook
 * (IQ1_S 16 KB, IQ2_S 8 KB).  IQ4_NL takes one fma per 32-element group instead
 * of one per block, so handing its sums through LDS would cost eight times as
 * much (34816 x 5120, one token: 83 against 44 us).
 *
 * walk_rows says which: the row walk pays from about 2700 rows per block of a
 * row on (block ranges / row walk: 65536 x 256, one and five tokens, Q3_K 12.2 /
 * 4.4 and 32.9 / 8.0 us, IQ1_S 17.2 / 7.7 and 45.4 / 11.3; 8192 x 768, five
 * tokens, Q3_K 6.4 / 5.7), up to as many blocks as where the codebook in LDS
 * or, from four tokens on, the shared activations win again (65536 x 1536 and
 * 65536 x 5120, one token, IQ2_S 41 / 39 and 96 / 127 us; 65536 x 1280 IQ1_S 27 /
 * 32, IQ2_S 36 / 33; 65536 x 5120 Q3_K 54 / 48; 65536 x 2048 and 65536 x 3072, five tokens, IQ2_S 78 / 73 and 98 / 108).
 * An IQ1_S walk of four to seven tokens is still 2 to 5 % behind the kernel
 * that stood here before the block ranges (65536 x 2048, five tokens 67 / 70). */
template <int T, int MT>
bool walk_rows(uint32_t rows, uint32_t nb)
{
    constexpr bool book = table_dwords<T>() > 0, gains = MT > 3 || T == kIQ2S || T == kIQ2XS;
    const uint32_t most = book ? (MT > 3 ? 6 : 4) + (gains && rows >= 65536 ? 2 : 0) : MT > 3 ? 10 : 20;
    return T == kIQ4NL || (nb <= most && rows >= 2700 * nb);
}

/* eight tokens: in the registers of eight wavefronts per SIMD the compiler
 * orders the loads one after another (Q5_K 65536 x 768 57 against 29 us) */
template <int T, int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, MT == 8 ? 6 : 8)))
void gemv_rows_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ x, float *__restrict__ y, uint32_t ldy,
                      uint32_t rows, uint32_t nb, const uint32_t *__restrict__ iq1s_grid)
{
    const int l = threadIdx.x & 7;
    const uint32_t row = (blockIdx.x * 256u + threadIdx.x) >> 3;
    const uint8_t *wr = w + (size_t)(row < rows ? row : rows - 1) * nb * block_bytes<T>();
    const uint32_t *table = table_of<T>(iq1s_grid);
    float acc[MT], scalar[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = scalar[t] = 0.0f;
    for (uint32_t b = 0; b < nb; ++b) {
        const uint8_t *blk = wr + (size_t)b * block_bytes<T>();
        LaneBlock lb;
        int m0 = 0, m1 = 0;
        decode_walk<T>(blk, l, table, lb, m0);
        if constexpr (T == kIQ1S) m1 = m0;
        else if constexpr (has_extra<T>()) extra_factors<T>(blk, l, m0, m1);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint8_t *xb = x + ((size_t)t * nb + b) * kQ8KBytes;
            const float xs = *reinterpret_cast<const float *>(xb);
            const int *aq = reinterpret_cast<const int *>(xb + 4) + l;
            if constexpr (T == kIQ4NL) {
#pragma unroll
                for (int g = 0; g < 8; ++g)
                    acc[t] = __builtin_fmaf(fmul_rn(lb.gd[g], xs), (float)dot4z((int)lb.q[g], aq[8 * g]), acc[t]);
                /* from five tokens on the compiler would move the links past
                 * the other tokens and keep their products in registers (eight
                 * tokens, 34816 x 5120: 353 against 117 us); below, its order
                 * is the faster one (three tokens, 17408 columns: 70 against
                 * 113 us) */
                if constexpr (MT > 4) asm volatile("" : "+v"(acc[t]));
            } else {
                int wsum = 0;
#pragma unroll
                for (int g = 0; g < 8; ++g) wsum = mad24(lb.s[g], dot4z((int)lb.q[g], aq[8 * g]), wsum);
                const float d = fmul_rn(lb.d, xs);
                acc[t] = __builtin_fmaf(d, (float)wsum, acc[t]);
                if constexpr (has_extra<T>()) {
                    const float extra = (float)row_extra(xb, l, m0, m1);
                    if constexpr (T == kIQ1S) scalar[t] = fadd_rn(scalar[t], fmul_rn(d, extra));
                    else scalar[t] = __builtin_fmaf(-fmul_rn(lb.dmin, xs), extra, scalar[t]);
                }
                if constexpr (MT > 3) {
                    if constexpr (has_extra<T>()) asm volatile("" : "+v"(acc[t]), "+v"(scalar[t]));
                    else asm volatile("" : "+v"(acc[t]));
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        float v = fadd_rn(acc[t], __shfl_xor(acc[t], 4, 64));
        v = fadd_rn(v, __shfl_xor(v, 2, 64));
        v = fadd_rn(v, __shfl_xor(v, 1, 64));
        if constexpr (T == kIQ1S) v = fadd_rn(v, fmul_rn(0.125f, scalar[t]));
        else if constexpr (has_extra<T>()) v = fadd_rn(v, scalar[t]);
        if (l == 0 && row < rows) y[(size_t)t * ldy + row] = v;
    }
}

template <int T, int MT, int H>
void launch_format_typed(const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows, uint32_t nb,
                         const void *grid, hipStream_t stream)
{
    const uint32_t *iq1s = static_cast<const uint32_t *>(grid);
    if constexpr (T != kIQ4NL) {
        if (!walk_rows<T, MT>(rows, nb)) {
            using F = GemvFormat<T, MT>;
            const uint32_t phases = (nb + F::kBlocks - 1) / F::kBlocks, blocks = (nb + phases - 1) / phases;
            hipLaunchKernelGGL((gemv_format_kernel<T, MT, H>), dim3((rows + 7) / 8), dim3(64 * H),
                               F::table + blocks * F::per_block, stream, w, x, y, ldy, rows, nb, blocks, iq1s);
            return;
        }
    }
    /* eight lanes per row in 32-bit thread numbers */
    constexpr uint32_t kRange = 1u << 28;
    for (uint32_t r = 0; r < rows; r += kRange) {
        const uint32_t n = rows - r < kRange ? rows - r : kRange;
        hipLaunchKernelGGL((gemv_rows_kernel<T, MT>), dim3((n + 31) / 32), dim3(256), 0, stream,
                           w + (size_t)r * nb * block_bytes<T>(), x, y + r, ldy, n, nb, iq1s);
        if (rows - r <= kRange) break;
    }
}

template <int T>
void launch_format_m(int m, const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows, uint32_t nb,
                     const void *grid, hipStream_t stream)
{
    switch (m) {
    case 1: launch_format_typed<T, 1, 8>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 2: launch_format_typed<T, 2, 8>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 3:
        if (nb < 40) launch_format_typed<T, 3, 8>(w, x, y, ldy, rows, nb, grid, stream);
        else launch_format_typed<T, 3, 12>(w, x, y, ldy, rows, nb, grid, stream);
        break;
    case 4: launch_format_typed<T, 4, 12>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 5: launch_format_typed<T, 5, 12>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 6: launch_format_typed<T, 6, 12>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 7: launch_format_typed<T, 7, 12>(w, x, y, ldy, rows, nb, grid, stream); break;
    default: launch_format_typed<T, 8, 12>(w, x, y, ldy, rows, nb, grid, stream); break;
    }
}
/* ---- row decode ------------------------------------------------------------ */

/* rows[r] of the matrix into out[r * width ..]; the row index of output row
 * r is ids[r] (a token id) when ids is set, else first + r.  One workgroup
 * per (block, output row); E threads = elements per block. */
template <int T, int E>
__global__ __launch_bounds__(256) void row_decode_kernel(const uint8_t *__restrict__ w, const uint32_t *__restrict__ ids,
                                                         uint32_t first, uint32_t limit, float *__restrict__ out,
                                                         uint32_t width, uint64_t row_bytes, uint32_t block_bytes)
{
    __shared__ int bad[256 / 64];
    const uint32_t b = blockIdx.x, r = blockIdx.y;
    uint32_t src = ids ? ids[r] : first + r;
    if (src >= limit) src = limit - 1;
    const uint8_t *blk = w + src * row_bytes + (size_t)b * block_bytes;
    const int i = threadIdx.x;
    float v = 0.0f;
    bool nonfinite = false;
    if (i < E) {
        v = element_weight<T>(blk, i);
        nonfinite = !__builtin_isfinite(v);
    }
    /* non-finite weights in the block: any other one makes this element NaN */
    const unsigned long long ballot = __ballot(nonfinite);
    if ((threadIdx.x & 63) == 0) bad[threadIdx.x >> 6] = __popcll(ballot);
    __syncthreads();
    if (i >= E) return;
    int count = 0;
    for (int k = 0; k < (E + 63) / 64; ++k) count += bad[k];
    /* inf * 0 on the x86 host the reference runs on gives the "indefinite"
     * quiet NaN, sign bit set */
    if (count - (nonfinite ? 1 : 0) > 0) v = __uint_as_float(0xffc00000u);
    else v = __fadd_rn(v, 0.0f);
    out[(size_t)r * width + (size_t)b * E + i] = v;
}

/* F32 / F16 / BF16 rows: copied or converted element by element */
template <int T>
__global__ __launch_bounds__(256) void row_convert_kernel(const uint8_t *__restrict__ w, const uint32_t *__restrict__ ids,
                                                          uint32_t first, uint32_t limit, float *__restrict__ out,
                                                          uint32_t width, uint64_t row_bytes)
{
    const uint32_t r = blockIdx.y, e = blockIdx.x * 256u + threadIdx.x;
    if (e >= width) return;
    uint32_t src = ids ? ids[r] : first + r;
    if (src >= limit) src = limit - 1;
    const uint8_t *row = w + src * row_bytes;
    float v;
    if constexpr (T == kF32) v = reinterpret_cast<const float *>(row)[e];
    else if constexpr (T == kF16) v = f16_to_f32(ld16(row + 2 * (size_t)e));
    else v = bf16_to_f32(ld16(row + 2 * (size_t)e));
    out[(size_t)r * width + e] = v;
}

__global__ __launch_bounds__(256) void fill_kernel(float *__restrict__ out, uint64_t count, float value)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i < count) out[i] = value;
}

}  // namespace

/* ---- host side --------------------------------------------------------------- */

void launch_fill_f32(float *out, uint64_t count, float value, hipStream_t stream)
{
    if (!count) return;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, out, count, value);
}

bool format_block_shape(int type, uint32_t *elements, uint32_t *bytes)
{
    uint32_t e = 256, b = 0;
    switch (type) {
    case kF32: e = 1; b = 4; break;
    case kF16: case kBF16: e = 1; b = 2; break;
    case kQ4_0: e = 32; b = 18; break;
    case kQ4_1: e = 32; b = 20; break;
    case kQ5_0: e = 32; b = 22; break;
    case kQ5_1: e = 32; b = 24; break;
    case kQ8_0: e = 32; b = 34; break;
    case kIQ4NL: e = 32; b = 18; break;
    case kQ2K: b = 84; break;
    case kQ3K: b = 110; break;
    case kQ4K: b = 144; break;
    case kQ5K: b = 176; break;
    case kQ6K: b = 210; break;
    case kIQ2XXS: b = 66; break;
    case kIQ2XS: b = 74; break;
    case kIQ2S: b = 82; break;
    case kIQ3XXS: b = 98; break;
    case kIQ3S: b = 110; break;
    case kIQ4XS: b = 136; break;
    case kIQ1S: b = 50; break;
    case kIQ1M: b = 56; break;
    default: return false;
    }
    *elements = e;
    *bytes = b;
    return true;
}

bool format_takes_q8k(int type)
{
    switch (type) {
    case kQ2K: case kQ3K: case kQ4K: case kQ5K: case kQ6K: case kIQ2XXS: case kIQ2XS: case kIQ2S: case kIQ3XXS:
    case kIQ3S: case kIQ4XS: case kIQ4NL: case kIQ1S: case kIQ1M: return true;
    default: return false;
    }
}

bool launch_gemm_format(int type, int m, const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows,
                        uint32_t nb, const void *grid, hipStream_t stream)
{
    if (m < 1 || m > 8 || ldy < rows || !rows || !nb) return false;
    switch (type) {
    case kQ2K: launch_format_m<kQ2K>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kQ3K: launch_format_m<kQ3K>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kQ5K: launch_format_m<kQ5K>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ2XXS: launch_format_m<kIQ2XXS>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ2XS: launch_format_m<kIQ2XS>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ2S: launch_format_m<kIQ2S>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ3XXS: launch_format_m<kIQ3XXS>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ3S: launch_format_m<kIQ3S>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ4XS: launch_format_m<kIQ4XS>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ4NL: launch_format_m<kIQ4NL>(m, w, x, y, ldy, rows, nb, grid, stream); return true;
    case kIQ1S:
        if (!grid) return false;
        launch_format_m<kIQ1S>(m, w, x, y, ldy, rows, nb, grid, stream);
        return true;
    default: return false;
    }
}

bool format_row_decodable(int type)
{
    switch (type) {
    case kF32: case kF16: case kBF16: case kQ8_0: case kIQ4NL: case kQ2K: case kQ3K: case kQ4K: case kQ5K: case kQ6K:
        return true;
    default: return false;
    }
}

bool launch_row_decode(int type, const uint8_t *w, const uint32_t *ids, uint32_t first, uint32_t count,
                       uint32_t limit, float *out, uint32_t width, hipStream_t stream)
{
    uint32_t e = 0, b = 0;
    if (!count || !limit || !format_block_shape(type, &e, &b) || width % e || !format_row_decodable(type))
        return false;
    const uint64_t row_bytes = (uint64_t)width / e * b;
    if (e == 1) {
        const dim3 grid((width + 255) / 256, count);
        switch (type) {
        case kF32: hipLaunchKernelGGL(row_convert_kernel<kF32>, grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes); break;
        case kF16: hipLaunchKernelGGL(row_convert_kernel<kF16>, grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes); break;
        default: hipLaunchKernelGGL(row_convert_kernel<kBF16>, grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes); break;
        }
        return true;
    }
    const dim3 grid(width / e, count);
    switch (type) {
    case kQ8_0: hipLaunchKernelGGL((row_decode_kernel<kQ8_0, 32>), grid, dim3(64), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    case kIQ4NL: hipLaunchKernelGGL((row_decode_kernel<kIQ4NL, 32>), grid, dim3(64), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    case kQ2K: hipLaunchKernelGGL((row_decode_kernel<kQ2K, 256>), grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    case kQ3K: hipLaunchKernelGGL((row_decode_kernel<kQ3K, 256>), grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    case kQ4K: hipLaunchKernelGGL((row_decode_kernel<kQ4K, 256>), grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    case kQ5K: hipLaunchKernelGGL((row_decode_kernel<kQ5K, 256>), grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    default: hipLaunchKernelGGL((row_decode_kernel<kQ6K, 256>), grid, dim3(256), 0, stream, w, ids, first, limit, out, width, row_bytes, b); break;
    }
    return true;
}

}  // namespace q38
