"""Times of calls that once lost to the kernels they replaced.  Each bound
lies between the two forms' times.  Best of several runs, GPU events."""
import ctypes

import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(300)]


def best_us(call, calls=40, runs=7):
    import torch
    call()
    best = 1e30
    for _ in range(runs):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        start.record()
        for _ in range(calls):
            call()
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end) / calls * 1e3)
    return best


def product(device, qtype, rows, width, tokens, fp32=False):
    """a product over random bytes: the time does not depend on the values"""
    import torch
    import q38hip
    from oracle import FORMATS
    elements, nbytes = FORMATS[qtype]
    lib = q38hip.lib()
    w = torch.randint(0, 120, (rows * (width // elements) * nbytes,), dtype=torch.uint8, device=device)
    x = torch.randn(tokens, width, device=device)
    x = x if fp32 else q38hip.quantize_q8_k(x)
    y = torch.empty(tokens, rows, device=device)
    tensor = q38hip.make_tensor(w.data_ptr(), qtype, width, rows, w.numel())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    entry = lib.q38hip_gemm_f32 if fp32 else lib.q38hip_gemm_q8_k
    args = (ctypes.c_void_p(y.data_ptr()), ctypes.c_void_p(x.data_ptr()), tokens, width, ctypes.byref(tensor), stream)
    keep = (w, x, y, tensor)

    def call():
        assert entry(*args) and keep
    return call


@pytest.mark.parametrize("name,rows,width,tokens,bound", (
    ("Q3_K", 65536, 256, 1, 7.5),       # 4.4 us; 11 with a workgroup per eight rows
    ("Q3_K", 65536, 256, 5, 20.0),      # 7.6; 30
    ("IQ1_S", 65536, 256, 5, 25.0),     # 11.3; 42
    ("IQ2_S", 248320, 256, 1, 50.0)))   # 25; 65
def test_short_rows(device, name, rows, width, tokens, bound):
    import oracle
    took = best_us(product(device, getattr(oracle, name), rows, width, tokens))
    print("%s %d x %d, %d tokens: %.1f us" % (name, rows, width, tokens, took), flush=True)
    assert took < bound


@pytest.mark.parametrize("name,rows,width,tokens,bound", (
    ("Q6_K", 1, 17408, 24, 155.0),      # 113 us in launches of eight; 197 in one
    ("IQ4_NL", 248320, 256, 9, 75.0),   # 48; 112
    ("Q5_K", 248320, 256, 9, 65.0)))    # 43; 91
def test_few_tokens_of_a_batch(device, name, rows, width, tokens, bound):
    import oracle
    took = best_us(product(device, getattr(oracle, name), rows, width, tokens))
    print("%s %d x %d, %d tokens: %.1f us" % (name, rows, width, tokens, took), flush=True)
    assert took < bound


def test_batch_against_its_launches(device):
    """24 tokens of Q6_K, 256 x 10240: no more than three launches of eight
    (90 us; 118 in one prompt launch)"""
    import oracle
    batch = best_us(product(device, oracle.Q6_K, 256, 10240, 24))
    eight = best_us(product(device, oracle.Q6_K, 256, 10240, 8))
    print("24 tokens %.1f us, 8 tokens %.1f us" % (batch, eight), flush=True)
    assert batch < 1.15 * 3 * eight


@pytest.mark.parametrize("name,rows,width,tokens,bound", (
    ("Q4_K", 96, 5120, 1, 120.0),       # 54 us; 267 with the elements of a quad decoded one by one
    ("Q4_K", 65536, 768, 2, 50.0),      # 19; 115
    ("Q5_K", 65536, 2048, 1, 160.0),    # 78; 325
    ("Q2_K", 65536, 2048, 1, 110.0),    # 42; 174
    ("IQ4_NL", 65536, 768, 1, 50.0)))   # 17; 92
def test_float_input(device, name, rows, width, tokens, bound):
    import oracle
    took = best_us(product(device, getattr(oracle, name), rows, width, tokens, fp32=True), calls=20)
    print("%s %d x %d, %d tokens, fp32 input: %.1f us" % (name, rows, width, tokens, took), flush=True)
    assert took < bound


def test_sample_few_of_many(device):
    """15.4 us; 31.7 by counting"""
    import torch
    import q38hip
    vocab = 1 << 20
    logits, token, state = torch.randn(vocab, device=device), torch.zeros(1, dtype=torch.int32, device=device), ctypes.c_uint64(5)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def call():
        assert q38hip.lib().q38hip_sample(ctypes.c_void_p(token.data_ptr()), ctypes.byref(state),
                                          ctypes.c_void_p(logits.data_ptr()), vocab, 0.7, 0.95, 0.0, 2, None, 0, stream)
    took = best_us(call)
    print("2 of %d logits: %.1f us" % (vocab, took), flush=True)
    assert took < 24.0


def test_attention_workspace(device):
    """A call whose buffers only together reach the size where an allocation
    gets dear takes what it takes with a little less to allocate: 131 and 130
    us, 157 with all buffers in one allocation."""
    import time
    import torch
    import q38hip
    rows = context = 64
    x = torch.randn(rows, 14336, device=device)
    norm, keys = torch.ones(256, device=device), torch.randn(context, 1024, device=device)
    values = torch.randn(1024, q38hip.value_pitch(context), device=device)
    out = torch.empty(rows, 6144, device=device)
    q8k = torch.empty(rows * 24 * 292, dtype=torch.uint8, device=device)
    p = [ctypes.c_void_p(a) for a in (out.data_ptr(), q8k.data_ptr(), x.data_ptr(), x.data_ptr() + 12288 * 4,
                                      x.data_ptr() + 13312 * 4, norm.data_ptr(), keys.data_ptr(), values.data_ptr())]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    best = {True: 1e30, False: 1e30}
    for _ in range(300):
        for with_q8k in best:
            torch.cuda.synchronize()
            start = time.perf_counter()
            assert q38hip.lib().q38hip_attention_rows(p[0], p[1] if with_q8k else None, p[2], p[3], p[4], 14336, p[5],
                                                      p[5], p[6], p[7], context, 0, rows, stream)
            best[with_q8k] = min(best[with_q8k], time.perf_counter() - start)
    print("with Q8_K output %.1f us, without %.1f us" % (best[True] * 1e6, best[False] * 1e6), flush=True)
    assert best[False] < 1.12 * best[True]
