"""Performance cases of the library's public entry points.

Four kinds of work, each through the entry points a program calls:

* linear:    fp32 activations in, one matrix or the matrices of one transformer
             block of the 27B shape, fp32 outputs.  Q8_K formats go through
             q38hip_quantize_q8_k and a q38hip_gemm_q8_k* call per matrix, float
             formats through q38hip_gemm_f32; the LM head adds q38hip_argmax.
* attention: q38hip_attention_rows over a filled cache.
* sample:    q38hip_sample over one row of logits.
* model:     a request through the model API: reset, prefill, then greedy tokens
             (plain or MTP speculative), the logits of every step returned.

Sizes are the model's (hidden 5120, FFN 17408, 24 heads of 256, 4 KV heads,
vocabulary 248320) or generic.  Every result of the library is defined bit for
bit (one order of every fp32 operation), so another correct implementation
gives the same bits: the tolerance is "exact" throughout.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3.8-27b-in-c_amd"))
import q38hip  # noqa: E402
from q38hip import synth  # noqa: E402
from q38hip.model import Model  # noqa: E402

# format: GGML type id, elements per block, bytes per block, byte offsets of the fp16 scales
FORMATS = {
    "f32": (0, 1, 4, ()), "f16": (1, 1, 2, ()), "bf16": (30, 1, 2, ()), "q8_0": (8, 32, 34, (0,)),
    "q2_k": (10, 256, 84, (80, 82)), "q3_k": (11, 256, 110, (108,)), "q4_k": (12, 256, 144, (0, 2)),
    "q5_k": (13, 256, 176, (0, 2)), "q6_k": (14, 256, 210, (208,)), "iq2_xxs": (16, 256, 66, (0,)),
    "iq2_xs": (17, 256, 74, (0,)), "iq3_xxs": (18, 256, 98, (0,)), "iq1_s": (19, 256, 50, (0,)),
    "iq4_nl": (20, 32, 18, (0,)), "iq3_s": (21, 256, 110, (0,)), "iq2_s": (22, 256, 82, (0,)),
    "iq4_xs": (23, 256, 136, (0,)), "iq1_m": (29, 256, 56, ()),
}
FLOAT_FORMATS = ("f32", "f16", "bf16", "q8_0")
IQ4NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)

HIDDEN, FFN, VOCAB = 5120, 17408, 248320
DELTANET = ((16480, HIDDEN), (HIDDEN, 6144), (2 * FFN, HIDDEN), (HIDDEN, FFN))
ATTENTION = ((14336, HIDDEN), (HIDDEN, 6144), (2 * FFN, HIDDEN), (HIDDEN, FFN))
SHAPES = {"deltanet": DELTANET, "attention": ATTENTION, "ffn": ATTENTION[2:], "head": ((VOCAB, HIDDEN),)}
Q8K = 292
MODEL_CONTEXT = 4608


def listed():
    return [
        # the DeltaNet beta / alpha projections, which GGUF writers leave in fp32: the smallest matrix of a decode step
        {"name": "ssm_f32", "kind": "linear", "format": "f32", "shape": "single", "rows": 96, "width": HIDDEN,
         "tokens": 1, "tiled": False},
        # one sampled token of a chat request, with the command line's default sampler settings
        {"name": "sample_top20", "kind": "sample", "vocab": VOCAB, "top_k": 20, "top_p": 0.95, "temperature": 1.0,
         "penalty": 0.0},
        # decode, one token: the matrices of a DeltaNet block of a Q4_K_M file
        {"name": "decode_q4k", "kind": "linear", "format": "q4_k", "shape": "deltanet", "tokens": 1, "tiled": True},
        # the MTP verify batch (draft length 3): the matrices of a full-attention block
        {"name": "verify_q4k", "kind": "linear", "format": "q4_k", "shape": "attention", "tokens": 3, "tiled": True},
        # decode, one token, of the smallest file format
        {"name": "decode_iq1m", "kind": "linear", "format": "iq1_m", "shape": "deltanet", "tokens": 1, "tiled": True},
        # the LM head over three verify rows, then the greedy tokens
        {"name": "head_q6k", "kind": "linear", "format": "q6_k", "shape": "head", "tokens": 3, "tiled": False},
        # decode, one token, of a Q5_K file: the FFN
        {"name": "decode_q5k", "kind": "linear", "format": "q5_k", "shape": "ffn", "tokens": 1, "tiled": False},
        # decode, one token, of a Q8_0 file: the matrices of a full-attention block
        {"name": "decode_q8_0", "kind": "linear", "format": "q8_0", "shape": "attention", "tokens": 1, "tiled": False},
        # a prompt of ragged length through the FFN of an IQ4_XS file
        {"name": "prompt_iq4xs", "kind": "linear", "format": "iq4_xs", "shape": "ffn", "tokens": 301, "tiled": False},
        # three verify rows of one full-attention layer at a 4K cache
        {"name": "attention_4k", "kind": "attention", "context": 5120, "position": 4099, "rows": 3},
        # a request to the Q4_K_M model: a prompt, then MTP speculative decoding
        {"name": "model_q4km", "kind": "model", "layout": "q4km", "prompt": 509, "steps": 12, "draft": 3},
        # a long prompt through the IQ1_M model and its first tokens
        {"name": "model_iq1m", "kind": "model", "layout": "iq1m", "prompt": 4096, "steps": 4, "draft": 3},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_linear(rng):
    name = rng.choice(sorted(FORMATS))
    tokens = rng.choice((1, 1, 1, 2, 3, 4, 5, _log(rng, 6, 512), _log(rng, 6, 512)))
    case = {"kind": "linear", "format": name, "tokens": tokens, "tiled": False}
    if name == "q4_k" or (name == "iq1_m" and tokens <= 8):
        case["tiled"] = rng.random() < 0.7
    shape = rng.choice(("deltanet", "attention", "ffn", "single", "single", "single"))
    case["shape"] = shape
    if shape == "single":
        case["rows"] = _log(rng, 48, 2 * FFN)
        step = 32 if FORMATS[name][1] < 256 and name in FLOAT_FORMATS else 256
        case["width"] = rng.choice((5120, 6144, 10240, 17408)) if case["tiled"] else step * max(1, _log(rng, 512, FFN) // step)
    return case


def draw(rng):
    kind = rng.choice(("linear",) * 6 + ("attention", "attention", "sample", "model"))
    if kind == "linear":
        return _draw_linear(rng)
    if kind == "attention":
        context = _log(rng, 64, 5120)
        rows = min(context, rng.choice((1, 2, 3, 4, 5, _log(rng, 6, 256))))
        return {"kind": "attention", "context": context, "position": rng.randint(0, context - rows), "rows": rows}
    if kind == "sample":
        return {"kind": "sample", "vocab": rng.choice((VOCAB, _log(rng, 30000, VOCAB))), "top_k": rng.choice((1, 20, 40, _log(rng, 5, 256))),
                "top_p": rng.choice((0.8, 0.95, 1.0)), "temperature": rng.choice((0.6, 0.7, 1.0)), "penalty": rng.choice((0.0, 1.5))}
    layout = rng.choice(("q4km", "iq1m"))
    return {"kind": "model", "layout": layout, "prompt": _log(rng, 8, 509 if layout == "q4km" else 4000),
            "steps": rng.randint(1, 4), "draft": rng.choice((0, 1, 2, 3))}


# ---- linear ------------------------------------------------------------------------------------------------------


def _matrices(case):
    return ((case["rows"], case["width"]),) if case["shape"] == "single" else SHAPES[case["shape"]]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _halves(g, count):
    """|N(0, 0.01)| in fp16, as bytes"""
    return torch.empty(count, device="cuda").normal_(0.0, 0.01, generator=g).abs_().half().view(torch.uint8).view(count, 2)


def _weights(name, rows, width, g):
    """a GGUF matrix of the format: random quants and scales, fp16 super-scales |N(0, 0.01)|"""
    _, elements, nbytes, fields = FORMATS[name]
    if elements == 1:
        w = torch.empty((rows, width), device="cuda").normal_(0.0, 0.02, generator=g)
        return w.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[name]).view(torch.uint8).reshape(-1)
    count = rows * (width // elements)
    data = torch.randint(0, 256, (count, nbytes), dtype=torch.uint8, device="cuda", generator=g)
    for at in fields:
        data[:, at:at + 2] = _halves(g, count)
    if name == "iq1_m":   # the fp16 super-scale lies in the high nibbles of the four scale words
        half = _halves(g, count)
        for k in range(4):
            nibble = (half[:, k // 2] >> (4 * (k % 2))) & 15
            data[:, 49 + 2 * k] = (data[:, 49 + 2 * k] & 15) | (nibble << 4)
    return data.reshape(-1)


def _activations(case, g):
    return [torch.empty((case["tokens"], width), device="cuda").normal_(0.0, 1.0, generator=g) for _, width in _matrices(case)]


def _prepare_linear(case, seed):
    g, lib, name, tokens = _generator(seed), q38hip.lib(), case["format"], case["tokens"]
    qtype = FORMATS[name][0]
    state = {"x": _activations(case, g), "keep": [], "calls": [], "out": []}
    for (rows, width), x in zip(_matrices(case), state["x"]):
        w = _weights(name, rows, width, g)
        y = torch.zeros((tokens, rows), device="cuda")
        if name in FLOAT_FORMATS:
            tensor = q38hip.make_tensor(w.data_ptr(), qtype, width, rows, w.numel())
            state["calls"].append((lib.q38hip_gemm_f32, (y.data_ptr(), x.data_ptr(), tokens, width, ctypes.byref(tensor))))
            state["keep"] += [w, tensor]
            state["out"].append(y)
            continue
        xq = torch.zeros(tokens * (width // 256) * Q8K, dtype=torch.uint8, device="cuda")
        state["calls"].append((lib.q38hip_quantize_q8_k, (xq.data_ptr(), x.data_ptr(), width, tokens)))
        if case["tiled"]:
            tiled = (q38hip.repack_q4k_tiles if name == "q4_k" else q38hip.repack_iq1m_tiles)(w, width, rows)
            call = lib.q38hip_gemm_q8_k_tiled if name == "q4_k" else lib.q38hip_gemm_q8_k_iq1m_tiled
            state["calls"].append((call, (y.data_ptr(), xq.data_ptr(), tokens, width, tiled.data_ptr(), rows)))
            state["keep"] += [tiled, xq]
        else:
            tensor = q38hip.make_tensor(w.data_ptr(), qtype, width, rows, w.numel())
            state["calls"].append((lib.q38hip_gemm_q8_k, (y.data_ptr(), xq.data_ptr(), tokens, width, ctypes.byref(tensor))))
            state["keep"] += [w, xq, tensor]
        state["out"].append(y)
    if case["shape"] == "head":
        best = torch.zeros(tokens, dtype=torch.int32, device="cuda")
        state["calls"].append((lib.q38hip_argmax, (best.data_ptr(), state["out"][0].data_ptr(), VOCAB, tokens)))
        state["out"].append(best)
    return state


def _run_linear(state):
    stream = torch.cuda.current_stream().cuda_stream
    for call, args in state["calls"]:
        if not call(*args, stream):
            raise RuntimeError(q38hip.last_error())
    return state["out"]


def _half(data, at):
    return data[:, at:at + 2].contiguous().view(torch.float16).double()


def _dequantise(name, data, width):
    """rows of a matrix in 64 bits; None for the formats with a codebook"""
    _, elements, nbytes, _ = FORMATS[name]
    if elements == 1:
        kind = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[name]
        return data.view(kind).double().view(-1, width)
    b = data.view(-1, nbytes)
    i = b.int()
    if name == "q8_0":
        return (_half(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()).view(-1, width)
    if name in ("q4_k", "q5_k"):
        p = i[:, 4:16]
        scale = torch.cat((p[:, 0:4] & 63, (p[:, 8:12] & 15) | (p[:, 0:4] >> 6) << 4), 1).double()
        low = torch.cat((p[:, 4:8] & 63, (p[:, 8:12] >> 4) | (p[:, 4:8] >> 6) << 4), 1).double()
        qs = i[:, nbytes - 128:].view(-1, 4, 1, 32)
        q = torch.cat((qs & 15, qs >> 4), 2).view(-1, 8, 32)
        if name == "q5_k":
            bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
            q = q + (((i[:, 16:48].view(-1, 1, 32) >> bit) & 1) << 4)
        w = (_half(b, 0) * scale).unsqueeze(2) * q.double() - (_half(b, 2) * low).unsqueeze(2)
        return w.reshape(-1, width)
    if name == "q6_k":
        ql, qh = i[:, :128].view(-1, 2, 2, 32), i[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat((ql & 15, ql >> 4), 2)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | high << 4) - 32
        scale = b[:, 192:208].contiguous().view(torch.int8).double() * _half(b, 208)
        return (q.double().view(-1, 16, 16) * scale.unsqueeze(2)).reshape(-1, width)
    if name == "iq4_xs":
        shift = 2 * torch.arange(8, device=b.device, dtype=torch.int32)
        high = ((i[:, 2] | i[:, 3] << 8).unsqueeze(1) >> shift) & 3
        low = torch.stack((i[:, 4:8] & 15, i[:, 4:8] >> 4), 2).view(-1, 8)
        qs = i[:, 8:].view(-1, 8, 16)
        q = torch.tensor(IQ4NL, device=b.device, dtype=torch.float64)[torch.cat((qs & 15, qs >> 4), 2).long()]
        return (q * (_half(b, 0) * ((low | high << 4) - 32).double()).unsqueeze(2)).reshape(-1, width)
    return None


def _q8k_values(x):
    """what the Q8_K blocks of x stand for, in 64 bits"""
    v = x.view(x.shape[0], -1, 256)
    at = v.abs().argmax(2, keepdim=True)
    inverse = -127.0 / v.gather(2, at)
    return (torch.clamp(torch.round(inverse * v), max=127.0).double() * (1.0 / inverse).double()).view(x.shape)


def _exact_linear(case, seed):
    name = case["format"]
    if name not in FLOAT_FORMATS + ("q4_k", "q5_k", "q6_k", "iq4_xs"):
        return None
    g, out = _generator(seed), []
    xs = _activations(case, g)
    for (rows, width), x in zip(_matrices(case), xs):
        data = _weights(name, rows, width, g).view(rows, -1)
        xd = x.double() if name in FLOAT_FORMATS else _q8k_values(x)
        y = [xd @ _dequantise(name, data[r:r + 4096].reshape(-1), width).T for r in range(0, rows, 4096)]
        out.append(torch.cat(y, 1))
    return out + [None] if case["shape"] == "head" else out


# ---- attention ---------------------------------------------------------------------------------------------------


def _prepare_attention(case, seed):
    g, context, rows = _generator(seed), case["context"], case["rows"]
    normal = lambda *shape: torch.empty(shape, device="cuda").normal_(0.0, 1.0, generator=g)  # noqa: E731
    state = {"position": case["position"], "in": normal(rows, 14336), "q_norm": 1.0 + 0.1 * normal(256), "k_norm": 1.0 + 0.1 * normal(256)}
    state["keys"], values = normal(context, 1024), normal(context, 1024)
    state["values"] = torch.zeros((1024, q38hip.value_pitch(context)), device="cuda")
    state["values"][:, :context] = values.T
    return state


def _run_attention(s):
    out, q8k = q38hip.attention_rows(s["in"], s["q_norm"], s["k_norm"], s["keys"], s["values"], s["position"])
    return [out, q8k, s["keys"], s["values"]]


def _exact_attention(case, seed):
    s, rows, at = _prepare_attention(case, seed), case["rows"], case["position"]
    x = s["in"].double()
    qg = x[:, :12288].view(rows, 24, 2, 256)
    end = at + rows

    def rotated(v, weight):
        v = v * torch.rsqrt(v.square().mean(2, keepdim=True) + 1e-6) * weight.double()
        pair = torch.arange(32, device="cuda", dtype=torch.float64)
        angle = torch.arange(at, end, device="cuda", dtype=torch.float64).view(-1, 1, 1) * 1e7 ** (-2.0 * pair / 64)
        a, b = v[..., :32].clone(), v[..., 32:64].clone()
        v[..., :32], v[..., 32:64] = a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()
        return v

    q = rotated(qg[:, :, 0].clone(), s["q_norm"])
    keys, values = s["keys"].double(), s["values"].double()
    keys[at:end] = rotated(x[:, 12288:13312].reshape(rows, 4, 256).clone(), s["k_norm"]).view(rows, 1024)
    values[:, at:end] = x[:, 13312:].T
    k, v = keys[:end].view(end, 4, 256), values[:, :end].view(4, 256, end)
    score = torch.einsum("thd,phd->thp", q, k.repeat_interleave(6, 1)) / 16.0
    seen = torch.arange(end, device="cuda").view(1, 1, -1) <= torch.arange(at, end, device="cuda").view(-1, 1, 1)
    weight = torch.softmax(score.masked_fill(~seen, -math.inf), 2)
    out = torch.einsum("thp,hdp->thd", weight, v.repeat_interleave(6, 0)) * torch.sigmoid(qg[:, :, 1])
    return [out.reshape(rows, 6144), None, keys, values]


# ---- sample ------------------------------------------------------------------------------------------------------


def _prepare_sample(case, seed):
    g = _generator(seed)
    logits = torch.empty(case["vocab"], device="cuda").normal_(0.0, 3.0, generator=g)
    seen = torch.zeros(case["vocab"], dtype=torch.uint8, device="cuda")
    seen[torch.randint(0, case["vocab"], (400,), device="cuda", generator=g)] = 1
    return {"logits": logits, "seen": seen if case["penalty"] else None, "case": case, "seed": int(seed)}


def _run_sample(s):
    c = s["case"]
    sampler = q38hip.Sampler(seed=s["seed"] + 1, temperature=c["temperature"], top_p=c["top_p"], presence_penalty=c["penalty"], top_k=c["top_k"])
    token = q38hip.sample(s["logits"], sampler, presence=s["seen"])
    return {"token": token, "state_low": sampler.state & 0xFFFFFFFF, "state_high": sampler.state >> 32}


# ---- model -------------------------------------------------------------------------------------------------------

_MODELS = {}


def _model(layout):
    """the open model of a layout (random-init 27B weights, MTP on), which a server keeps for all its requests"""
    if layout not in _MODELS:
        path = synth.model_path(1, layout)
        if path is None:
            raise RuntimeError("no directory has room for the synthetic %s model" % layout)
        model = Model.open(synth.write_model_gguf(path, 1, layout), MODEL_CONTEXT)
        model.enable_mtp()
        _MODELS[layout] = model
    return _MODELS[layout]


def _prepare_model(case, seed):
    prompt = np.random.default_rng(int(seed)).integers(0, VOCAB, size=case["prompt"]).astype(np.uint32)
    return {"model": _model(case["layout"]), "prompt": prompt, "steps": case["steps"], "draft": case["draft"]}


def _run_model(s):
    model = s["model"]
    model.reset()
    rows, tokens = [model.prefill(s["prompt"])], []
    for _ in range(s["steps"]):
        token = int(rows[-1].argmax())
        if s["draft"]:
            accepted, row = model.speculative_greedy(token, VOCAB - 1, s["draft"])
            tokens += [int(t) for t in accepted]
        else:
            row = model.forward_token(token)
            tokens.append(token)
        rows.append(row)
    return [np.stack(rows), np.array(tokens, dtype=np.int64)]


def _model_bytes(layout):
    """weights of (the 64 blocks, the MTP block with its input projection, the LM head)"""
    unit = {"q4km": 144, "iq1m": 56}[layout] / 256
    size = lambda shapes: sum(rows * width for rows, width in shapes)  # noqa: E731
    blocks = 48 * size(DELTANET) + 16 * size(ATTENTION)
    return blocks * unit, (size(ATTENTION) + HIDDEN * 2 * HIDDEN) * unit, VOCAB * HIDDEN * 210 / 256


# ---- the cases' interface ----------------------------------------------------------------------------------------


def prepare(case, seed):
    return {"kind": case["kind"], "state": _KINDS[case["kind"]][0](case, seed)}


def run(state):
    return _KINDS[state["kind"]][1](state["state"])


def exact(case, seed):
    if case["kind"] == "linear":
        return _exact_linear(case, seed)
    return _exact_attention(case, seed) if case["kind"] == "attention" else None


def tolerance(case):
    return "exact"


def work(case):
    kind = case["kind"]
    if kind == "linear":
        _, elements, nbytes, _ = FORMATS[case["format"]]
        bytes_, flops = 0, 0
        for rows, width in _matrices(case):
            bytes_ += rows * (width // elements) * nbytes + 4 * case["tokens"] * (width + rows)
            flops += 2 * rows * width * case["tokens"]
        return {"bytes": bytes_, "flops": flops}
    if kind == "attention":
        rows, end = case["rows"], case["position"] + case["rows"]
        pairs = rows * case["position"] + rows * (rows + 1) // 2
        return {"bytes": 8 * 1024 * end + rows * (14336 * 4 + 6144 * 4 + 24 * Q8K), "flops": 4 * 24 * 256 * pairs}
    if kind == "sample":
        return {"bytes": case["vocab"] * (5 if case["penalty"] else 4), "flops": 0}
    blocks, mtp, head = _model_bytes(case["layout"])
    parameters = 48 * sum(r * w for r, w in DELTANET) + 16 * sum(r * w for r, w in ATTENTION)
    step = blocks + head + case["draft"] * (mtp + head)
    rows = case["prompt"] + case["steps"] * max(1, case["draft"])
    return {"bytes": blocks + head + case["steps"] * step, "flops": 2 * parameters * rows}


_KINDS = {"linear": (_prepare_linear, _run_linear), "attention": (_prepare_attention, _run_attention),
          "sample": (_prepare_sample, _run_sample), "model": (_prepare_model, _run_model)}
