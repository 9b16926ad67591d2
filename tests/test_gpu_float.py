"""Matrices against fp32 activations (q38hip_gemm_f32) at the edges of the
kernel's 64-row workgroups, 64-column stages and token tiles, against the
oracle's one-token chain (orc_format_gemv_f32).  Bar: bit-identical outputs,
the chain having one order.  F32, F16 and BF16 take any width; an infinite
weight or activation must reach exactly its own outputs."""
import numpy as np
import pytest

import format_cases as fc
from oracle import BF16, F16, F32, FORMAT_NAMES, IQ4_NL, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]

# (rows, width, tokens); widths are rounded up to the format's block
SHAPES = ((1, 1, 1), (63, 67, 2), (65, 130, 3), (64, 64, 4), (5, 255, 5), (70, 320, 9), (66, 1000, 33), (64, 192, 66),
          (96, 5120, 1), (130, 769, 1))


def run(device, oracle, qtype, rows, width, tokens, data, x):
    import torch
    import q38hip
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    got = q38hip.gemm_f32(dev(data), qtype, width, rows, dev(x)).cpu().numpy()
    want = np.stack([oracle.gemv_f32(qtype, data, rows, x[t]) for t in range(tokens)])
    finite = np.isfinite(want)
    assert np.array_equal(finite, np.isfinite(got)) and np.array_equal(np.isnan(want), np.isnan(got))
    assert int((got.view(np.uint32) != want.view(np.uint32))[~np.isnan(want)].sum()) == 0


@pytest.mark.parametrize("qtype", (F32, F16, BF16, Q8_0, IQ4_NL, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K),
                         ids=lambda t: FORMAT_NAMES[t])
def test_float_gemm_edges(device, oracle, qtype):
    rng = np.random.default_rng(900 + qtype)
    elements = fc.FORMATS[qtype][0]
    for rows, width, tokens in SHAPES:
        width = -(-width // elements) * elements
        print("%s rows=%d width=%d tokens=%d" % (FORMAT_NAMES[qtype], rows, width, tokens), flush=True)
        data = fc.random_matrix(qtype, rows, width, rng)
        run(device, oracle, qtype, rows, width, tokens, data, rng.standard_normal((tokens, width)).astype(np.float32))


@pytest.mark.parametrize("qtype", (F32, F16, BF16, Q8_0, IQ4_NL, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K),
                         ids=lambda t: FORMAT_NAMES[t])
def test_float_gemm_tall(device, oracle, qtype):
    """Above 16384 rows, where up to eight tokens take stages of 64 columns
    (below, most take 128), and from 65536 rows on, where short rows of some
    formats are walked by a lane each."""
    rng = np.random.default_rng(920 + qtype)
    elements = fc.FORMATS[qtype][0]
    for rows, width, counts in ((16450, 67, (1, 2, 3, 4, 7)), (16385, 321, (1, 2, 3, 5)), (65601, 130, (1, 2, 3))):
        width = -(-width // elements) * elements
        data = fc.random_matrix(qtype, rows, width, rng)
        x = rng.standard_normal((max(counts), width)).astype(np.float32)
        for tokens in counts:
            print("%s rows=%d width=%d tokens=%d" % (FORMAT_NAMES[qtype], rows, width, tokens), flush=True)
            run(device, oracle, qtype, rows, width, tokens, data, x[:tokens])


@pytest.mark.parametrize("qtype", (F32, F16, BF16), ids=lambda t: FORMAT_NAMES[t])
def test_float_gemm_non_finite(device, oracle, qtype):
    rng = np.random.default_rng(950 + qtype)
    rows, width, tokens = 67, 131, 5
    data = fc.random_matrix(qtype, rows, width, rng)
    bits = {F32: (np.uint32, 0x7F800000), F16: (np.uint16, 0x7C00), BF16: (np.uint16, 0x7F80)}[qtype]
    cells = data.view(bits[0]).reshape(rows, width)
    cells[3, 130], cells[66, 0] = bits[1], bits[1]
    x = rng.standard_normal((tokens, width)).astype(np.float32)
    x[2, 64], x[4, 130] = -np.inf, np.nan
    run(device, oracle, qtype, rows, width, tokens, data, x)


def test_float_gemm_row_ranges(device, oracle):
    """Rows of 64 MiB: sixty-four of them pass a workgroup's 32-bit offsets, so
    the matrix runs in ranges of 63 rows."""
    import torch
    import q38hip
    rows, width = 65, (1 << 24) + 4
    g = torch.Generator(device=device)
    g.manual_seed(41)
    w = torch.empty((rows, width), device=device).normal_(0.0, 1.0, generator=g)
    x = torch.empty((1, width), device=device).normal_(0.0, 1.0, generator=g)
    got = q38hip.gemm_f32(w.view(torch.uint8).reshape(-1), F32, width, rows, x).cpu().numpy()[0]
    host = x[0].cpu().numpy()
    for row in (0, 62, 63, 64):
        want = oracle.gemv_f32(F32, w[row].cpu().numpy().view(np.uint8), 1, host)
        assert got[row:row + 1].view(np.uint32)[0] == np.asarray(want, np.float32).view(np.uint32)[0], row


def test_float_gemm_token_ranges(device):
    """More token tiles than a grid has: two launches.  Rows of one column, so
    that an output is one product, rounded once."""
    import torch
    import q38hip
    rows, tokens = 2, 65535 * 64 + 3
    g = torch.Generator(device=device)
    g.manual_seed(42)
    w = torch.empty(rows, device=device).normal_(0.0, 1.0, generator=g)
    x = torch.empty((tokens, 1), device=device).normal_(0.0, 1.0, generator=g)
    got = q38hip.gemm_f32(w.view(torch.uint8), F32, 1, rows, x)
    assert torch.equal(got, x * w.view(1, rows))
