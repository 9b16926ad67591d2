/* GEMV / small-M GEMM and row decode for the remaining
 * GGUF matrix formats of the reference model (src/qwen38/qwen38_model.c:
 * 172-189): Q2_K, Q3_K, Q5_K, IQ2_XXS, IQ2_XS, IQ2_S, IQ3_XXS, IQ3_S,
 * IQ4_XS, IQ4_NL, IQ1_S against Q8_K activations.
 *
 * Q8_K path.  Each of the reference's AVX2 kernels (qwen38_quant.c:510-1253,
 * 1636-1725) keeps eight fp32 lanes per row; for every super-block, lane l
 * gets d * W[l], where W[l] is the exact integer sum over bytes 4l..4l+3 of
 * each 32-element group, each group-half scaled by its integer sub-block
 * scale.  Here eight GPU lanes own a row's eight accumulator lanes (a
 * wavefront holds eight rows): each decodes the four weights of each group
 * it needs into a packed int8 dword (grid value and sign folded in),
 * multiplies with v_dot4_i32_i8 against the activation dword, scales, and
 * runs its fmaf chain.  The eight lanes then add in the reference's tree
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

/* y[t * ldy + row] for t < MT: eight rows per wavefront, eight lanes per row */
template <int T, int MT>
__global__ __launch_bounds__(256) void gemv_format_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ x,
                                                          float *__restrict__ y, uint32_t ldy, uint32_t rows,
                                                          uint32_t nb, const uint32_t *__restrict__ iq1s_grid)
{
    const int lane = threadIdx.x & 63, l = lane & 7;
    const uint32_t row = (blockIdx.x * 256u + threadIdx.x) >> 3;
    const uint32_t r = row < rows ? row : rows - 1;
    const uint32_t bytes = block_bytes<T>();
    const uint8_t *wr = w + (size_t)r * nb * bytes;
    float acc[MT], scalar[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = scalar[t] = 0.0f;

    for (uint32_t b = 0; b < nb; ++b) {
        const uint8_t *blk = wr + (size_t)b * bytes;
        LaneBlock lb;
        decode_lane<T>(blk, l, iq1s_grid, lb);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint8_t *xb = x + ((size_t)t * nb + b) * kQ8KBytes;
            const float xs = *reinterpret_cast<const float *>(xb);
            const uint32_t *aq = reinterpret_cast<const uint32_t *>(xb + 4);
            if constexpr (T == kIQ4NL) {
#pragma unroll
                for (int g = 0; g < 8; ++g) {
                    const int wg = dot4z((int)lb.q[g], (int)aq[8 * g + l]);
                    acc[t] = __builtin_fmaf(__fmul_rn(lb.gd[g], xs), (float)wg, acc[t]);
                }
            } else {
                int wsum = 0;
#pragma unroll
                for (int g = 0; g < 8; ++g) wsum += lb.s[g] * dot4z((int)lb.q[g], (int)aq[8 * g + l]);
                const float d = __fmul_rn(lb.d, xs);
                acc[t] = __builtin_fmaf(d, (float)wsum, acc[t]);
                if constexpr (T == kQ2K || T == kQ5K) {
                    const float dmin = __fmul_rn(lb.dmin, xs);
                    scalar[t] = __builtin_fmaf(-dmin, (float)block_extra<T>(blk, xb), scalar[t]);
                } else if constexpr (T == kIQ1S) {
                    scalar[t] = __fadd_rn(scalar[t], __fmul_rn(d, (float)block_extra<T>(blk, xb)));
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        /* ((a0 + a4) + (a2 + a6)) + ((a1 + a5) + (a3 + a7)), qwen38_quant.c:303-310 */
        float v = __fadd_rn(acc[t], __shfl_xor(acc[t], 4, 64));
        v = __fadd_rn(v, __shfl_xor(v, 2, 64));
        v = __fadd_rn(v, __shfl_xor(v, 1, 64));
        if constexpr (T == kIQ1S) v = __fadd_rn(v, __fmul_rn(0.125f, scalar[t]));
        else if constexpr (has_extra<T>()) v = __fadd_rn(v, scalar[t]);
        if (l == 0 && row < rows) y[(size_t)t * ldy + row] = v;
    }
}

template <int T, int MT>
void launch_format_typed(const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows, uint32_t nb,
                         const void *grid, hipStream_t stream)
{
    hipLaunchKernelGGL((gemv_format_kernel<T, MT>), dim3((rows + 31) / 32), dim3(256), 0, stream, w, x, y, ldy, rows,
                       nb, static_cast<const uint32_t *>(grid));
}

template <int T>
void launch_format_m(int m, const uint8_t *w, const uint8_t *x, float *y, uint32_t ldy, uint32_t rows, uint32_t nb,
                     const void *grid, hipStream_t stream)
{
    switch (m) {
    case 1: launch_format_typed<T, 1>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 2: launch_format_typed<T, 2>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 3: launch_format_typed<T, 3>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 4: launch_format_typed<T, 4>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 5: launch_format_typed<T, 5>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 6: launch_format_typed<T, 6>(w, x, y, ldy, rows, nb, grid, stream); break;
    case 7: launch_format_typed<T, 7>(w, x, y, ldy, rows, nb, grid, stream); break;
    default: launch_format_typed<T, 8>(w, x, y, ldy, rows, nb, grid, stream); break;
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
