"""The single-launch kernels report their own launch's status: an error that
earlier HIP work left on the calling thread is neither taken for theirs (the
call would be refused, or would fall to launches of eight tokens) nor cleared."""
import ctypes

import numpy as np
import pytest

import format_cases as fc
from oracle import F16, F32, Q3_K, Q5_K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype,tokens", ((F32, 1), (F16, 9), (Q5_K, 24), (Q3_K, 70)),
                         ids=("F32-1", "F16-9", "Q5_K-24", "Q3_K-70"))
def test_earlier_error_is_left_alone(device, oracle, qtype, tokens):
    import torch
    import q38hip
    lib = q38hip.lib()
    rng = np.random.default_rng(31)
    rows, width = 70, 512
    data = fc.random_matrix(qtype, rows, width, rng)
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    if qtype in (F32, F16):
        call, host_in = lib.q38hip_gemm_f32, x
        want = np.stack([oracle.gemv_f32(qtype, data, rows, x[t]) for t in range(tokens)])
    else:
        call, host_in = lib.q38hip_gemm_q8_k, oracle.quantize(x.reshape(-1)).view(np.uint8)
        blocks = host_in.view(np.uint8).reshape(tokens, -1)
        want = np.stack([oracle.gemv(qtype, data, rows, b.copy().view(oracle.quantize(x[0]).dtype)) for b in blocks])
    w, xd = torch.from_numpy(data).to(device), torch.from_numpy(host_in).to(device)
    out = torch.zeros((tokens, rows), device=device)
    tensor = q38hip.make_tensor(w.data_ptr(), qtype, width, rows, w.numel())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    lib.hipGetLastError()
    try:
        assert lib.hipSetDevice(1 << 20) != 0          # no such device
        left = lib.hipPeekAtLastError()
        ok = call(ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(xd.data_ptr()), tokens, width,
                  ctypes.byref(tensor), stream)
        after = lib.hipPeekAtLastError()
    finally:
        lib.hipGetLastError()                          # nothing is left for torch to find
    assert left != 0
    assert ok, q38hip.last_error()
    assert after == left
    got = out.cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.astype(np.float32).view(np.uint32))
