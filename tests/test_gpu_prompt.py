"""Prompt batches (9 tokens and more) of the row-major Q8_K formats on the
matrix cores (q38hip_gemm_q8_k) against the oracle's one-token GEMV.  Bar:
bit-identical fp32 outputs, since every integer sum is exact and the fp32
chains keep their order.  Shapes sit at the edges of the 64-row x 64-token
workgroup; the second input is Q8_K blocks with the extremes of the int8 and
int16 fields and of the weights' packed fields, where the sums are largest."""
import numpy as np
import pytest

import format_cases as fc
from oracle import FORMAT_NAMES, IQ1_M, IQ1_S, IQ4_NL, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8K_DTYPE, Q8K_FORMATS

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]

TYPES = [t for t in Q8K_FORMATS if t != IQ1_M]


def check(device, oracle, qtype, rows, width, data, q8, tokens):
    import torch
    import q38hip
    nb = width // 256
    want = np.stack([oracle.gemv(qtype, data, rows, q8[t * nb:(t + 1) * nb]) for t in range(tokens)])
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    got = q38hip.gemm_q8_k(dev(data), qtype, width, rows, dev(q8.view(np.uint8)), tokens).cpu().numpy()
    wrong = int((got.view(np.uint32) != want.astype(np.float32).view(np.uint32)).sum())
    assert wrong == 0, "%d of %d differ" % (wrong, got.size)


@pytest.mark.parametrize("qtype", TYPES, ids=lambda t: FORMAT_NAMES[t])
def test_prompt_batches_match_oracle(device, oracle, qtype):
    rng = np.random.default_rng(700 + qtype)
    # at most 128 row tiles and three tiles of 64 tokens are two rounds of the
    # chip, or one of 128-token workgroups: the last two shapes run those
    for rows, width, tokens in ((1, 256, 24), (63, 512, 64), (65, 1280, 65), (130, 5120, 33), (64, 768, 131),
                                (4100, 256, 9), (8200, 256, 130), (8190, 256, 130), (8130, 768, 131)):
        print("%s rows=%d width=%d tokens=%d" % (FORMAT_NAMES[qtype], rows, width, tokens), flush=True)
        data = fc.random_matrix(qtype, rows, width, rng)
        q8 = oracle.quantize(rng.standard_normal(tokens * width).astype(np.float32))
        check(device, oracle, qtype, rows, width, data, q8, tokens)


@pytest.mark.parametrize("qtype", TYPES, ids=lambda t: FORMAT_NAMES[t])
@pytest.mark.parametrize("rows,tokens", ((40, 26), (8150, 129)))
def test_prompt_extreme_fields_match_oracle(device, oracle, qtype, rows, tokens):
    rng = np.random.default_rng(800 + qtype)
    width = 512
    data = fc.random_matrix(qtype, rows, width, rng).reshape(rows, -1)
    scales = fc.random_matrix(qtype, rows, width, rng).reshape(rows, -1)
    data[:20][data[:20] < 128] = 0      # rows of 0x00 and 0xff bytes
    data[:20][data[:20] >= 128] = 255
    fields = np.zeros(data.shape[1], bool)
    block = fc.FORMATS[qtype][1]
    for at in fc.SCALE_FIELDS[qtype]:   # finite super-scales in every row
        for start in range(0, data.shape[1], block):
            fields[start + at:start + at + 2] = True
    data[:, fields] = scales[:, fields]
    q8 = np.zeros(tokens * width // 256, dtype=Q8K_DTYPE)
    q8["scale"] = rng.uniform(-0.1, 0.1, q8.size)
    q8["quants"] = rng.choice([-128, -127, 127], q8["quants"].shape)
    q8["quants"][:8] = 127              # whole blocks of one sign: the largest sums
    q8["quants"][8:16] = -128
    q8["sums"] = rng.choice([-32768, -2048, -1, 63, 2047, 32767], q8["sums"].shape)
    check(device, oracle, qtype, rows, width, data.reshape(-1), q8, tokens)


@pytest.mark.parametrize("qtype", (Q2_K, Q4_K, Q5_K, IQ1_S), ids=lambda t: FORMAT_NAMES[t])
def test_prompt_sums_of_one_sign_match_oracle(device, oracle, qtype):
    """Blocks whose sixteen sums lie at one end of int16: the min or correction
    sum of a block is then at its largest (Q5_K: 16 x 63 x 32768, twice 2^24),
    and is rounded once, when it becomes a float.  Some rows have the largest
    multipliers; the sums differ in their low bits, so that a sum that is
    rounded on the way shows."""
    rng = np.random.default_rng(850 + qtype)
    rows, width, tokens = 70, 768, 37
    data = fc.random_matrix(qtype, rows, width, rng).reshape(rows, -1)
    if qtype in (Q4_K, Q5_K):
        block = fc.FORMATS[qtype][1]
        for start in range(0, data.shape[1], block):
            data[:35, start + 4:start + 16] |= rng.integers(240, 256, (35, 12), dtype=np.uint8)
    q8 = np.zeros(tokens * width // 256, dtype=Q8K_DTYPE)
    q8["scale"] = rng.uniform(-0.1, 0.1, q8.size)
    q8["quants"] = rng.integers(-127, 128, q8["quants"].shape)
    q8["sums"] = 32767 - rng.integers(0, 200, q8["sums"].shape)
    q8["sums"][::2] = rng.integers(0, 200, q8["sums"][::2].shape) - 32768
    check(device, oracle, qtype, rows, width, data.reshape(-1), q8, tokens)


@pytest.mark.parametrize("qtype,rows,width,line", (
    (Q6_K, 512, 5120, 26), (Q6_K, 1000, 2048, 24), (Q6_K, 4700, 256, 10), (Q6_K, 1, 10496, 40), (Q4_K, 1, 10496, 25),
    (Q3_K, 16400, 256, 16), (IQ4_NL, 16390, 512, 12), (IQ1_S, 16390, 512, 12)))
def test_either_side_of_few_token_limit(device, oracle, qtype, rows, width, line):
    """the last batch that runs as launches of up to eight tokens, and the
    first of one launch"""
    rng = np.random.default_rng(880 + qtype)
    data = fc.random_matrix(qtype, rows, width, rng)
    q8 = oracle.quantize(rng.standard_normal((line + 1) * width).astype(np.float32))
    for tokens in (line, line + 1):
        check(device, oracle, qtype, rows, width, data, q8[:tokens * width // 256], tokens)
