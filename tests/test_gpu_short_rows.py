"""Few-token products (q38hip_gemm_q8_k, 1 to 8 tokens) of short rows, where a
matrix has many rows to a block of columns and eight lanes walk a row instead
of sharing its blocks, against the oracle's GEMV.  Bar: bit-identical outputs.
Rows lie on both sides of the line between the two (2700 rows per block, up to
4 to 20 blocks) and end inside a workgroup of 32 rows and of 8; the longest ones
take several phases through LDS, of a size that depends on the token count."""
import numpy as np
import pytest

import format_cases as fc
from oracle import FORMAT_NAMES, IQ1_M, Q4_K, Q6_K, Q8K_FORMATS

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]

TYPES = [t for t in Q8K_FORMATS if t not in (IQ1_M, Q4_K, Q6_K)]


@pytest.mark.parametrize("qtype", TYPES, ids=lambda t: FORMAT_NAMES[t])
def test_short_rows_match_oracle(device, oracle, qtype):
    import torch
    import q38hip
    rng = np.random.default_rng(600 + qtype)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    for rows, width in ((2699, 256), (2700, 256), (8111, 768), (10801, 1024), (13501, 1280), (43, 17408)):
        nb = width // 256
        data = fc.random_matrix(qtype, rows, width, rng)
        q8 = oracle.quantize(rng.standard_normal(8 * width).astype(np.float32))
        want = np.stack([oracle.gemv(qtype, data, rows, q8[t * nb:(t + 1) * nb]) for t in range(8)]).astype(np.float32)
        w, x = dev(data), dev(q8.view(np.uint8))
        for tokens in range(1, 9):
            print("%s rows=%d width=%d tokens=%d" % (FORMAT_NAMES[qtype], rows, width, tokens), flush=True)
            got = q38hip.gemm_q8_k(w, qtype, width, rows, x[:tokens * nb * 292], tokens).cpu().numpy()
            assert np.array_equal(got.view(np.uint32), want[:tokens].view(np.uint32)), (rows, width, tokens)
