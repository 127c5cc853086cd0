"""Workloads of the quantized-linear framework as a user's program runs them, through its public entry points: single
linears and MLP blocks called eagerly, decoder stacks stepping one token (replayed from a HIP graph as the greedy loops
do, or eagerly as transformers' generate() does) and reading prompts, and weights being converted at load time.

A case is a dict of plain values; `listed()` names the ones that are timed by default, `draw(rng)` gives others of the
same ranges.  `prepare` makes what the program holds before the call, `run` is one pass, `work` what the pass cannot do
without, `tolerance` how far another correct implementation of the same precision may be away.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tpp-pytorch-extension_amd"))

import tpp_pytorch_extension  # noqa: E402,F401
from tpp_pytorch_extension._C import _fused_llm_infer as fused  # noqa: E402
from tpp_pytorch_extension._C import _qtype as qtype  # noqa: E402
from tpp_pytorch_extension.llm import fused_gptj_infer as gptj  # noqa: E402
from tpp_pytorch_extension.llm import fused_llama_infer as llama  # noqa: E402
from tpp_pytorch_extension.llm import fused_opt_infer as opt  # noqa: E402
from tpp_pytorch_extension.llm import fused_qwen2_infer as qwen2  # noqa: E402

BF16 = torch.bfloat16
VOCAB = 32000
MAX_POSITIONS = 4096

# family, hidden, MLP width, query heads, key heads, head size
SHAPES = {
    "llama-7b": ("llama", 4096, 11008, 32, 32, 128),
    "llama-70b": ("llama", 8192, 28672, 64, 8, 128),
    "qwen2-7b": ("qwen2", 3584, 18944, 28, 4, 128),
    "gptj-6b": ("gptj", 4096, 16384, 16, 16, 256),
    "opt-2.7b": ("opt", 2560, 10240, 32, 32, 80),
}


def listed():
    return [
        # the smallest call: one MXFP4 projection of a batch of 16 (latency and launch cost)
        {"name": "fc_plain mxfp4 16 rows", "kind": "linear", "op": "fc_plain", "fmt": "mxfp4", "act": "bf16",
         "rows": 16, "n": 4096, "k": 4096},
        # W8A8 down-projection with its residual at the largest decode batch of the headline workload
        {"name": "fc_add qint8 64 rows", "kind": "linear", "op": "fc_add", "fmt": "qint8", "act": "bf16",
         "rows": 64, "n": 4096, "k": 11008},
        # SwiGLU block of a decode step of 50 sequences (an odd batch), MXFP4
        {"name": "swiglu_mlp mxfp4 50 rows", "kind": "mlp", "fmt": "mxfp4", "rows": 50, "hidden": 4096, "inter": 11008},
        # the same block in the W4A8 layout (USE_MXFP4_INT8) for a batch of 32
        {"name": "swiglu_mlp w4a8 32 rows", "kind": "mlp", "fmt": "w4a8", "rows": 32, "hidden": 4096, "inter": 11008},
        # loading a model: a blocked bf16 weight to MXFP4 and back to float
        {"name": "load mxfp4 11008 x 4096", "kind": "load", "fmt": "mxfp4", "n": 11008, "k": 4096},
        # greedy decoding of one sequence, 2048 keys in the cache, step replayed from its graph
        {"name": "decode llama-7b batch 1", "kind": "decode", "shape": "llama-7b", "fmt": "mxfp4", "layers": 4,
         "batch": 1, "context": 2048, "graph": True},
        # the same for 16 sequences
        {"name": "decode llama-7b batch 16", "kind": "decode", "shape": "llama-7b", "fmt": "mxfp4", "layers": 4,
         "batch": 16, "context": 2048, "graph": True},
        # an eager decode step (transformers' generate()) of another family: LayerNorm, pairwise rotary, 256-wide heads
        {"name": "decode gptj-6b batch 4 eager", "kind": "decode", "shape": "gptj-6b", "fmt": "qint8", "layers": 4,
         "batch": 4, "context": 700, "graph": False},
        # a prompt of a few hundred tokens (odd length)
        {"name": "prompt llama-7b mxfp4 333", "kind": "prompt", "shape": "llama-7b", "fmt": "mxfp4", "layers": 4,
         "batch": 1, "tokens": 333, "past": 0},
        # W8A8 prompt
        {"name": "prompt llama-7b qint8 1000", "kind": "prompt", "shape": "llama-7b", "fmt": "qint8", "layers": 4,
         "batch": 1, "tokens": 1000, "past": 0},
        # long prompt on unquantized weights, the front-ends' default
        {"name": "prompt llama-7b bf16 2048", "kind": "prompt", "shape": "llama-7b", "fmt": "bf16", "layers": 4,
         "batch": 1, "tokens": 2048, "past": 0},
        # the largest: a 70B-shape layer over a long prompt, grouped-query attention
        {"name": "prompt llama-70b mxfp4 2048", "kind": "prompt", "shape": "llama-70b", "fmt": "mxfp4", "layers": 2,
         "batch": 1, "tokens": 2048, "past": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "decode", "decode", "prompt", "prompt", "load"])
    if kind == "linear":
        fmt = rng.choice(["mxfp4", "qint8", "qint4", "qint2", "w4a8", "bf16"])
        act = rng.choice(["bf16", "bf16", "bf16", "f32", "f16"]) if fmt != "w4a8" else "bf16"
        return {"kind": "linear", "op": rng.choice(["fc_plain", "fc_add", "fc_silu"]) if act == "bf16" else "fc_plain",
                "fmt": fmt, "act": act, "rows": _log_int(rng, 1, 2048 if act == "bf16" else 512),
                "n": 64 * _log_int(rng, 16, 172), "k": 256 * _log_int(rng, 4, 43)}
    if kind == "mlp":
        return {"kind": "mlp", "fmt": rng.choice(["mxfp4", "qint8", "w4a8"]), "rows": _log_int(rng, 1, 2048),
                "hidden": 256 * rng.randint(8, 20), "inter": 256 * rng.randint(20, 64)}
    if kind == "decode":
        batch = _log_int(rng, 1, 48)
        return {"kind": "decode", "shape": rng.choice(["llama-7b", "llama-7b", "qwen2-7b", "gptj-6b", "opt-2.7b"]),
                "fmt": rng.choice(["mxfp4", "mxfp4", "qint8", "bf16"]), "layers": rng.randint(1, 4), "batch": batch,
                "context": _log_int(rng, 30, 4000 if batch <= 16 else 1500), "graph": rng.random() < 0.6}
    if kind == "prompt":
        batch = rng.choice([1, 1, 1, 2, 3])
        return {"kind": "prompt", "shape": rng.choice(["llama-7b", "llama-7b", "qwen2-7b", "gptj-6b", "opt-2.7b"]),
                "fmt": rng.choice(["mxfp4", "mxfp4", "qint8", "bf16"]), "layers": rng.randint(1, 4), "batch": batch,
                "tokens": _log_int(rng, 20, 2048 // batch), "past": rng.choice([0, 0, rng.randint(1, 1000)])}
    return {"kind": "load", "fmt": rng.choice(["mxfp4", "qint8", "qint2"]), "n": 64 * _log_int(rng, 16, 500),
            "k": 256 * _log_int(rng, 4, 43)}


# ----------------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _blocked(g, n, k, std=0.02):
    """A blocked bf16 weight [N/16][K/64][32][16][2], as FixLinear makes it."""
    w = (torch.randn((n, k), generator=g, device="cuda") * std).to(BF16)
    return w.view(n // 16, 16, k // 64, 32, 2).permute(0, 2, 3, 1, 4).contiguous()


def _int4(w):
    """A QINT4 weight: the VNNI2 layout with 256-wide blocks, [N/16][K/256][128][16][2]."""
    n, k = w.shape[0] * 16, w.shape[1] * 64
    return qtype.quantize_int4sym(w.view(n // 16, k // 256, 4, 32, 16, 2).reshape(n // 16, k // 256, 128, 16, 2), 256, 2, True)


QUANTIZE = {
    "mxfp4": qtype.remap_and_quantize_mxfp4,
    "qint8": qtype.remap_and_quantize_qint8,
    "qint4": _int4,
    "qint2": qtype.remap_and_quantize_qint2_intlv,
    "w4a8": lambda w: qtype.remap_and_quantize_mxfp4(w, True),
    "bf16": lambda w: w,
}


def _weight(g, fmt, n, k):
    return QUANTIZE[fmt](_blocked(g, n, k))


def _acts(g, *shape, dtype=BF16):
    """N(0, 1) activations whose channels differ in size, as behind a normalisation with its gamma."""
    gain = torch.exp(0.4 * torch.randn(shape[-1], generator=g, device="cuda"))
    return (torch.randn(shape, generator=g, device="cuda") * gain).to(dtype)


def _vec(g, n, dtype=BF16, std=0.1, mean=0.0):
    return (mean + std * torch.randn(n, generator=g, device="cuda")).to(dtype)


def _layers(g, case):
    family, hidden, inter, nq, nkv, head = SHAPES[case["shape"]]
    fmt = case["fmt"]

    def lin(n, k):
        return _weight(g, fmt, n, k)

    made = []
    for i in range(case["layers"]):
        q, k, v, o = lin(nq * head, hidden), lin(nkv * head, hidden), lin(nkv * head, hidden), lin(hidden, nq * head)
        if family in ("llama", "qwen2"):
            table = llama.llama_rotary_table(MAX_POSITIONS, head)
            norm = [_vec(g, hidden, torch.float32, mean=1.0) for _ in range(2)]
            mlp = [lin(inter, hidden), lin(inter, hidden), lin(hidden, inter)]
            if family == "llama":
                made.append(llama.LlamaDecoderLayer([norm[0], q, k, v, o, norm[1], *mlp, table], i, 1e-5, head,
                                                    MAX_POSITIONS, head))
            else:
                biases = [_vec(g, nq * head), _vec(g, nkv * head), _vec(g, nkv * head)]
                made.append(qwen2.Qwen2DecoderLayer([norm[0], q, k, v, o, norm[1], *mlp, *biases, table], i, 1e-6, head,
                                                    MAX_POSITIONS, head))
        elif family == "gptj":
            table = gptj.create_sinusoidal_positions(MAX_POSITIONS, 64).cuda()
            made.append(gptj.GPTJBlock([_vec(g, hidden, mean=1.0), _vec(g, hidden), q, k, v, o, lin(inter, hidden),
                                        _vec(g, inter), lin(hidden, inter), _vec(g, hidden), table], i, 1e-5, head,
                                       MAX_POSITIONS, 64))
        else:
            made.append(opt.OPTDecoderLayer([_vec(g, hidden, mean=1.0), _vec(g, hidden), _vec(g, hidden, mean=1.0),
                                             _vec(g, hidden), q, _vec(g, nq * head), k, _vec(g, nkv * head), v,
                                             _vec(g, nkv * head), o, _vec(g, hidden), lin(inter, hidden), _vec(g, inter),
                                             lin(hidden, inter), _vec(g, hidden)], i, 1e-5, 1e-5, head, True))
    return made


def _filled(g, case, capacity, context):
    _, _, _, _, nkv, head = SHAPES[case["shape"]]
    cache = llama.TppCache(capacity)
    for i in range(case["layers"]):
        kv = (case["batch"], nkv, context, head)
        cache.fill_(i, torch.randn(kv, generator=g, device="cuda", dtype=BF16),
                    torch.randn(kv, generator=g, device="cuda", dtype=BF16))
    return cache


def _logits(state, hidden):
    """Final norm and lm_head of the last position, as the front-ends' models end."""
    hidden = hidden[:, -1:].contiguous()
    if state["beta"] is None:
        hidden = llama.rms_norm(hidden, state["gamma"], 1e-5)
    else:
        hidden = gptj.lyr_norm(hidden, state["gamma"], state["beta"], 1e-5)
    return fused.fc_plain(hidden, state["lm_head"], None)


def _forward(state, cache):
    hidden = state["hidden"]
    for layer in state["layers"]:
        inputs = [hidden, state["mask"]] if isinstance(layer, opt.OPTDecoderLayer) else [hidden, state["mask"], state["pos"]]
        hidden = layer.forward(inputs, cache)[0]
    return hidden, _logits(state, hidden)


def _model(g, case):
    family, hidden = SHAPES[case["shape"]][:2]
    rms = family in ("llama", "qwen2")
    return {"layers": _layers(g, case), "gamma": _vec(g, hidden, torch.float32 if rms else BF16, mean=1.0),
            "beta": None if rms else _vec(g, hidden), "lm_head": _weight(g, case["fmt"], VOCAB, hidden), "mask": None}


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        act = {"bf16": BF16, "f16": torch.float16, "f32": torch.float32}[case["act"]]
        return {"op": case["op"], "w": _weight(g, case["fmt"], n, k), "x": _acts(g, m, k, dtype=act), "bias": _vec(g, n, act),
                "residual": _acts(g, m, n, dtype=act)}
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"op": "mlp", "gate": _weight(g, case["fmt"], i, h), "up": _weight(g, case["fmt"], i, h),
                "down": _weight(g, case["fmt"], h, i), "x": _acts(g, case["rows"], h), "residual": _acts(g, case["rows"], h)}
    if kind == "load":
        return {"op": "load", "fmt": case["fmt"], "w": _blocked(g, case["n"], case["k"])}
    hidden = SHAPES[case["shape"]][1]
    state = _model(g, case)
    state["op"], batch = kind, case["batch"]
    if kind == "decode":
        context = case["context"]
        state["hidden"] = _acts(g, batch, 1, hidden)
        state["pos"] = torch.full((batch, 1), context, dtype=torch.int64, device="cuda")
        # room for the tokens still to come, as a generation loop allocates it
        state["cache"], state["context"] = _filled(g, case, context + 128, context), context
        if case["graph"]:
            _forward(state, state["cache"])
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                state["out"] = _forward(state, state["cache"])
            torch.cuda.synchronize()
        return state
    tokens, past = case["tokens"], case["past"]
    state["hidden"] = _acts(g, batch, tokens, hidden)
    state["capacity"], state["past"] = past + tokens + 128, past
    state["cache"] = _filled(g, case, state["capacity"], past) if past else None
    state["pos"] = torch.arange(past, past + tokens, dtype=torch.int64, device="cuda").unsqueeze(0)
    if batch > 1:  # prompts of different length, padded on the left
        keep = torch.ones((batch, past + tokens), dtype=BF16, device="cuda")
        for b in range(1, batch):
            keep[b, :(past + tokens) * b // (4 * batch)] = 0
        state["mask"] = llama.TppCache(state["capacity"]).align_and_invert_mask(keep)
    return state


def run(state):
    op = state["op"]
    if op == "fc_plain":
        return torch.ops.tpp_llm.fc_plain(state["x"], state["w"], state["bias"], -1, [])
    if op == "fc_add":
        return torch.ops.tpp_llm.fc_add(state["x"], state["w"], state["bias"], state["residual"], 1.0)
    if op == "fc_silu":
        return torch.ops.tpp_llm.fc_silu(state["x"], state["w"], state["bias"])
    if op == "mlp":
        return torch.ops.tpp_llm.swiglu_mlp(state["x"], state["gate"], state["up"], state["down"], state["residual"], 1.0)
    if op == "load":
        q = QUANTIZE[state["fmt"]](state["w"])
        return [q.qdata, q.scales, q.dequantize()]
    if op == "decode":
        if "graph" in state:
            state["graph"].replay()
            hidden, logits = state["out"]
        else:
            hidden, logits = _forward(state, state["cache"])
        at = state["context"]
        return [hidden, logits, [[k[:, :, at], v[:, :, at]] for k, v in state["cache"].layers.values()]]
    cache = state["cache"]
    if cache is None:  # a new request: a cache of its own
        cache = llama.TppCache(state["capacity"])
    hidden, logits = _forward(state, cache)
    if not state["past"]:
        cache.advance(hidden.shape[1])
        return [hidden, logits, [cache.get(i) for i in range(len(state["layers"]))]]
    at = slice(state["past"], state["past"] + hidden.shape[1])
    return [hidden, logits, [[k[:, :, at], v[:, :, at]] for k, v in cache.layers.values()]]


BYTES_PER_WEIGHT = {"mxfp4": 0.5 + 1 / 32, "w4a8": 0.5 + 1 / 32, "qint8": 1 + 4 / 256, "qint4": 0.5 + 4 / 256,
                    "qint2": 0.25 + 4 / 256, "bf16": 2.0}


def work(case):
    kind = case["kind"]
    per = BYTES_PER_WEIGHT[case["fmt"]]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        a = 4 if case["act"] == "f32" else 2
        return {"bytes": per * n * k + a * (m * k + n + m * n * (2 if case["op"] == "fc_add" else 1)), "flops": 2.0 * m * n * k}
    if kind == "mlp":
        m, h, i = case["rows"], case["hidden"], case["inter"]
        return {"bytes": 3 * per * h * i + 6 * m * h, "flops": 6.0 * m * h * i}
    if kind == "load":
        return {"bytes": case["n"] * case["k"] * (2 + per + 4), "flops": 0.0}
    family, hidden, inter, nq, nkv, head = SHAPES[case["shape"]]
    b = case["batch"]
    s, past = (1, case["context"]) if kind == "decode" else (case["tokens"], case["past"])
    weights = hidden * (2 * nq + 2 * nkv) * head + hidden * inter * (3 if family in ("llama", "qwen2") else 2)
    keys = s * past + s * (s + 1) / 2
    layer = {"bytes": per * weights + 2.0 * 2 * b * nkv * head * (past + s), "flops": 2.0 * b * s * weights + 4.0 * b * nq * head * keys}
    return {"bytes": case["layers"] * layer["bytes"] + per * VOCAB * hidden + 2.0 * b * (2 * s * hidden + VOCAB),
            "flops": case["layers"] * layer["flops"] + 2.0 * b * VOCAB * hidden}


def tolerance(case):
    """About four times what was measured: linears against the same product in float64 (bf16 out 1.7e-3, half 2.1e-4,
    float 1.9e-6), stacks of up to four layers against themselves with another kernel family's summation order (1.1e-2;
    3.6e-2 where every linear quantizes its activations to int8, which turns a rounding flip into a step of the code)."""
    kind = case["kind"]
    if kind == "load":
        return "exact"
    if kind == "linear":
        return {"rel": {"bf16": 7e-3, "f16": 8e-4, "f32": 8e-6}[case["act"]]}
    if kind == "mlp":
        return {"rel": 1e-2}
    return {"rel": 0.12 if case["fmt"] == "qint8" else 4e-2}
