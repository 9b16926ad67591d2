/* C ABI of the full-attention decode core (declared in include/q38hip.h):
 * the kernels the engine runs for a full-attention block, callable on their
 * own for kernel-level parity tests and external callers. */
#include <hip/hip_runtime.h>

#include <cstring>
#include <vector>

#include "q38hip.h"
#include "q38_kernels.h"

namespace {

constexpr uint32_t kQGDim = 12288, kQDim = 6144, kKVDim = 1024, kHeads = 24;

/* The call's device buffers, released at its end: one allocation, or one per
 * buffer where only their sum reaches kLargeBytes.  From that size on hipMalloc
 * and hipFree take 23 us a pair, below it they are served from a pool in 1.4
 * us (64 rows of a 64-position context without Q8_K output, 2.4 MB in all: 157
 * us a call in one allocation, 131 in three). */
class Workspace {
public:
    static constexpr int kBuffers = 3;
    explicit Workspace(const size_t (&bytes)[kBuffers])
    {
        constexpr size_t kLargeBytes = (size_t)2 << 20;
        size_t total = 0, largest = 0;
        for (size_t n : bytes) {
            total += n;
            largest = n > largest ? n : largest;
        }
        const bool apart = total >= kLargeBytes && largest < kLargeBytes;
        size_t at = 0;
        for (int i = 0; i < kBuffers; ++i) {
            const size_t need = apart ? bytes[i] : i ? 0 : total;
            if (need && hipMalloc(&owned_[i], need) != hipSuccess) {
                owned_[i] = nullptr;
                ok_ = false;
                return;
            }
            buffer_[i] = static_cast<uint8_t *>(apart ? owned_[i] : owned_[0]) + (apart ? 0 : at);
            at += bytes[i];
        }
    }
    ~Workspace()
    {
        for (void *p : owned_)
            if (p) (void)hipFree(p);
    }
    Workspace(const Workspace &) = delete;
    Workspace &operator=(const Workspace &) = delete;
    bool ok() const { return ok_; }
    uint8_t *operator[](int i) const { return buffer_[i]; }

private:
    void *owned_[kBuffers] = {};
    uint8_t *buffer_[kBuffers] = {};
    bool ok_ = true;
};

constexpr size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

}  // namespace

extern "C" int q38hip_attention_rows(float *attention, Q38Q8KBlock *attention_q8k, const float *q_and_gate,
                                     const float *key, const float *value, uint64_t in_stride, const float *q_norm,
                                     const float *k_norm, float *key_cache, float *value_cache,
                                     uint32_t context_length, uint32_t position, uint32_t rows, void *stream)
{
    if (!attention || !q_and_gate || !key || !value || !q_norm || !k_norm || !key_cache || !value_cache || !rows ||
        !context_length)
        return q38::abi_fail("bad attention arguments");
    if (in_stride < kKVDim || (rows > 1 && in_stride < kQGDim)) return q38::abi_fail("row stride too small");
    if ((uint64_t)position + rows > context_length) return q38::abi_fail("position + rows beyond the context");
    if (context_length > q38::kMaxAttentionContext) return q38::abi_fail("context length above 524256 positions");
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone)
        return q38::abi_fail("stream synchronisation failed");
    /* The host side bounds a call of few rows, so it is kept to one
     * workspace, one upload and the RoPE rows of the call's own positions
     * (three rows at a 4K cache: 83 us a call; with the RoPE table of all 5120
     * positions of the context, five allocations and two uploads 1005 us). */
    const size_t rope_bytes = align256((size_t)rows * 64 * sizeof(float) + sizeof(uint32_t));
    const size_t q_bytes = align256((size_t)rows * kQDim * sizeof(float));
    const size_t score_bytes = align256((size_t)rows * kHeads * context_length * sizeof(float));
    const size_t out_bytes = attention_q8k ? 0 : (size_t)rows * kHeads * sizeof(Q38Q8KBlock);
    /* the RoPE rows, then the position word */
    std::vector<float> table((size_t)rows * 64 + 1);
    q38::rope_table_host(table.data(), position, rows);
    std::memcpy(&table[(size_t)rows * 64], &position, sizeof(position));
    Workspace work({rope_bytes + q_bytes, score_bytes, out_bytes});
    if (!work.ok()) return q38::abi_fail("device allocation failed");
    float *rope = reinterpret_cast<float *>(work[0]);
    uint32_t *pos = reinterpret_cast<uint32_t *>(rope + (size_t)rows * 64);
    float *q_buf = reinterpret_cast<float *>(work[0] + rope_bytes);
    float *scores = reinterpret_cast<float *>(work[1]);
    uint8_t *q_out = attention_q8k ? reinterpret_cast<uint8_t *>(attention_q8k) : work[2];
    if (hipMemcpyAsync(rope, table.data(), table.size() * sizeof(float), hipMemcpyHostToDevice, s) != hipSuccess ||
        !q38::configure_attention((int)context_length)) {
        (void)hipStreamSynchronize(s);
        return q38::abi_fail("attention set-up failed");
    }
    /* the kernels index the table by absolute position */
    const float *rope0 = reinterpret_cast<const float *>(reinterpret_cast<uintptr_t>(rope) -
                                                         (uintptr_t)position * 64 * sizeof(float));
    q38::launch_attention(attention, q_out, q_buf, q_and_gate, key, value, (long long)in_stride, q_norm, k_norm, rope0,
                          key_cache, value_cache, scores, (int)context_length, pos, (int)rows, s);
    const hipError_t launched = hipGetLastError();
    const hipError_t done = hipStreamSynchronize(s);
    if (launched != hipSuccess || done != hipSuccess) return q38::abi_fail("attention kernels failed");
    return 1;
}
