"""Performance cases: the work that programs give this framework, through its
public entry points.

  gemv      Runtime.gemv: one matrix-vector product, bf16 or fp16, packed or
            with a row pitch
  gemm      Runtime.gemm: one matrix product, bf16 or fp16
  decode    Engine.decode: forced tokens one by one behind a prompt, with the
            logits read back after the last (a program that samples itself)
  chat      Engine.generate: prompt and greedy reply in one call
  prompt    Engine.generate for the first token only: the prompt forms

Engines are loaded from a checkpoint directory that is written from the seed
and removed again. All model shapes have the head and row sizes of the
framework's presets; `layers` cuts the depth (with the 4096-entry vocabulary
of the "small" preset), so that most model cases are a few layers.
"""
import json
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

import xpu_playground_amd as xpu
from xpu_playground_amd import qwen3

DTYPES = {"bf16": (xpu.BF16, torch.bfloat16), "fp16": (xpu.FP16, torch.float16)}

# hidden, intermediate, query heads, kv heads: the presets' shapes
SHAPES = {"0.6b": (1024, 3072, 16, 8), "8b": (4096, 12288, 32, 8)}
FULL = {"layers": 28, "vocab": 151936}  # the whole qwen3-0.6b
CUT = {"vocab": 4096}  # the "small" preset's vocabulary
HEAD_DIM, EPS, THETA = 128, 1e-6, 1e6


def listed():
    return [
        # one projection of a small model: launch latency counts
        {"name": "gemv_small", "kind": "gemv", "dtype": "bf16", "m": 1024, "k": 1024, "lda": 1024},
        # odd sizes and a row pitch: a slice of a larger matrix
        {"name": "gemv_ragged", "kind": "gemv", "dtype": "bf16", "m": 5003, "k": 3001, "lda": 3005},
        # the headline benchmark's matrix: far past every cache
        {"name": "gemv_large", "kind": "gemv", "dtype": "fp16", "m": 16384, "k": 16384, "lda": 16384},
        # a few requests' rows against one weight matrix
        {"name": "gemm_few_rows", "kind": "gemm", "dtype": "bf16", "m": 24, "n": 4096, "k": 4096},
        # a product that cannot fill the chip with large tiles
        {"name": "gemm_mid", "kind": "gemm", "dtype": "bf16", "m": 1024, "n": 1024, "k": 1024},
        # the benchmark's ragged product
        {"name": "gemm_ragged", "kind": "gemm", "dtype": "fp16", "m": 3000, "n": 4097, "k": 2050},
        # the benchmark's square product
        {"name": "gemm_large", "kind": "gemm", "dtype": "bf16", "m": 4096, "n": 4096, "k": 4096},
        # the whole small model: a short question and a short greedy reply
        {"name": "chat_short", "kind": "chat", "shape": "0.6b", **FULL, "prompt": 32, "new": 32},
        # tokens behind a long context (a document in the prompt)
        {"name": "decode_long", "kind": "decode", "shape": "0.6b", "layers": 4, **CUT, "prompt": 2100, "steps": 8},
        # the whole small model reads the benchmark's prompt, default form
        {"name": "prompt_default", "kind": "prompt", "shape": "0.6b", **FULL, "prompt": 128, "form": "batched"},
        # a long prompt of an odd length, default form
        {"name": "prompt_default_long", "kind": "prompt", "shape": "0.6b", "layers": 4, **CUT, "prompt": 1531,
         "form": "batched"},
        # a long prompt on the matrix cores, the fast form
        {"name": "prompt_gemm", "kind": "prompt", "shape": "0.6b", "layers": 8, **CUT, "prompt": 2048,
         "form": "gemm"},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "gemm", "decode", "prompt", "prompt"])
    dtype = rng.choice(["bf16", "fp16"])
    if kind == "gemv":
        m, k = _log(rng, 64, 16384), _log(rng, 64, 16384)
        if rng.random() < 0.5:  # sizes of models are round, others are not
            m, k = (m + 63) // 64 * 64, (k + 63) // 64 * 64
        return {"kind": kind, "dtype": dtype, "m": m, "k": k, "lda": k + rng.choice([0, 0, 3, 64])}
    if kind == "gemm":
        m, n, k = _log(rng, 4, 4096), _log(rng, 64, 4096), _log(rng, 64, 4096)
        if rng.random() < 0.5:
            n, k = (n + 63) // 64 * 64, (k + 63) // 64 * 64
        return {"kind": kind, "dtype": dtype, "m": m, "n": n, "k": k}
    if kind == "decode":
        shape = rng.choice(["0.6b", "0.6b", "8b"])
        layers = rng.randint(1, 4 if shape == "0.6b" else 2)
        return {"kind": kind, "shape": shape, "layers": layers, **CUT,
                "prompt": _log(rng, 2, 4000 if shape == "0.6b" else 400), "steps": rng.randint(4, 12)}
    form = rng.choice(["batched", "batched", "gemm"])
    shape = "0.6b" if form == "batched" else rng.choice(["0.6b", "0.6b", "8b"])
    return {"kind": kind, "shape": shape, "layers": rng.randint(1, 4) if shape == "0.6b" else 1, **CUT,
            "prompt": _log(rng, 2, 2048), "form": form}


# ---------------------------------------------------------------- inputs

_rt = None


def _runtime():
    """The one runtime of the program."""
    global _rt
    if _rt is None:
        _rt = xpu.Runtime()
    return _rt


def _generator(seed, *more):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + sum(v * 7919 ** i for i, v in enumerate(more, 1))) % (1 << 62))
    return g


def _uniform(shape, dtype, seed, which):
    """U[-1, 1), the benchmark's data."""
    x = torch.rand(shape, generator=_generator(seed, which), device="cuda", dtype=torch.float32)
    return (2 * x - 1).to(dtype)


def _weights(case, seed):
    """The checkpoint's tensors by name: matrices N(0, 0.02^2), gains 1 + N(0, 0.1^2)."""
    hidden, inter, heads, kv = SHAPES[case["shape"]]
    sizes = {"self_attn.q_proj": (heads * HEAD_DIM, hidden), "self_attn.k_proj": (kv * HEAD_DIM, hidden),
             "self_attn.v_proj": (kv * HEAD_DIM, hidden), "self_attn.o_proj": (hidden, heads * HEAD_DIM),
             "self_attn.q_norm": (HEAD_DIM,), "self_attn.k_norm": (HEAD_DIM,),
             "mlp.gate_proj": (inter, hidden), "mlp.up_proj": (inter, hidden), "mlp.down_proj": (hidden, inter),
             "input_layernorm": (hidden,), "post_attention_layernorm": (hidden,)}
    names = [("model.layers.%d.%s.weight" % (i, n), s) for i in range(case["layers"]) for n, s in sizes.items()]
    names += [("model.embed_tokens.weight", (case["vocab"], hidden)), ("model.norm.weight", (hidden,))]
    g, out = _generator(seed, 11), {}
    for name, size in names:
        w = torch.randn(size, generator=g, device="cuda", dtype=torch.float32)
        out[name] = (1 + 0.1 * w if len(size) == 1 else 0.02 * w).to(torch.bfloat16)
    return out


def _write_checkpoint(path, case, weights):
    hidden, inter, heads, kv = SHAPES[case["shape"]]
    config = {"model_type": "qwen3", "hidden_act": "silu", "torch_dtype": "bfloat16", "hidden_size": hidden,
              "intermediate_size": inter, "num_hidden_layers": case["layers"], "num_attention_heads": heads,
              "num_key_value_heads": kv, "head_dim": HEAD_DIM, "vocab_size": case["vocab"], "rms_norm_eps": EPS,
              "rope_theta": THETA, "tie_word_embeddings": True}
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(config, f)
    header, at = {}, 0
    for name, w in weights.items():
        header[name] = {"dtype": "BF16", "shape": list(w.shape), "data_offsets": [at, at + w.numel() * 2]}
        at += w.numel() * 2
    text = json.dumps(header).encode()
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for w in weights.values():
            f.write(w.view(torch.int16).cpu().numpy().data)


def _engine(case, seed):
    need = case["prompt"] + case.get("new", 1) + case.get("steps", 0)
    path = tempfile.mkdtemp(prefix="qwen3_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    try:
        _write_checkpoint(path, case, _weights(case, seed))
        eng = qwen3.Engine(model_dir=path, max_seq=max(256, 1 << (need - 1).bit_length()), runtime=_runtime())
    finally:
        shutil.rmtree(path)
    if case.get("form") == "gemm":
        eng.set_prefill("gemm")
    return eng


def _tokens(case, seed):
    """The prompt, and for decode the forced tokens behind it."""
    n = case["prompt"] + case.get("steps", 0)
    return np.random.RandomState(seed % (1 << 31)).randint(0, case["vocab"], n).astype(np.uint32)


def prepare(case, seed):
    s = {"case": case}
    if case["kind"] in ("gemv", "gemm"):
        code, dtype = DTYPES[case["dtype"]]
        s.update(rt=_runtime(), code=code)
        if case["kind"] == "gemv":
            s["a"] = _uniform((case["m"], case["lda"]), dtype, seed, 1)
            s["b"] = _uniform((case["k"],), dtype, seed, 2)
            s["c"] = torch.empty(case["m"], dtype=dtype, device="cuda")
        else:
            s["a"] = _uniform((case["m"], case["k"]), dtype, seed, 1)
            s["b"] = _uniform((case["k"], case["n"]), dtype, seed, 2)
            s["c"] = torch.empty((case["m"], case["n"]), dtype=dtype, device="cuda")
        torch.cuda.synchronize()  # the runtime has its own stream
        return s
    s["engine"], s["tokens"] = _engine(case, seed), _tokens(case, seed)
    if case["kind"] == "decode":
        s["engine"].generate(s["tokens"][: case["prompt"]], 1, stop_on_eos=False)  # fills the KV caches
    return s


# ---------------------------------------------------------------- one pass

def _bf16(codes):
    return torch.from_numpy(codes.view(np.int16)).view(torch.bfloat16)


def run(state):
    c = state["case"]
    if c["kind"] == "gemv":
        state["rt"].gemv(state["code"], state["a"].data_ptr(), state["b"].data_ptr(), state["c"].data_ptr(), c["m"],
                         c["k"], c["lda"])
        return state["c"]
    if c["kind"] == "gemm":
        state["rt"].gemm(state["code"], state["a"].data_ptr(), state["b"].data_ptr(), state["c"].data_ptr(), c["m"],
                         c["n"], c["k"])
        return state["c"]
    eng, tokens, p = state["engine"], state["tokens"], c["prompt"]
    if c["kind"] == "decode":
        chosen = [eng.decode(int(tokens[p + i]), p + i) for i in range(c["steps"])]
        return {"tokens": np.array(chosen, np.int64), "logits": _bf16(eng.logits()), "hidden": _bf16(eng.hidden())}
    chosen, _, _ = eng.generate(tokens, c.get("new", 1), stop_on_eos=False)
    return {"tokens": chosen.astype(np.int64), "logits": _bf16(eng.logits()), "hidden": _bf16(eng.hidden())}


# ---------------------------------------------------------------- bounds

def work(case):
    if case["kind"] == "gemv":
        m, k = case["m"], case["k"]
        return {"bytes": 2 * (m * k + k + m), "flops": 2 * m * k}
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    hidden, inter, heads, kv = SHAPES[case["shape"]]
    layer = hidden * HEAD_DIM * (2 * heads + 2 * kv) + 3 * hidden * inter  # weights of one layer
    head = hidden * case["vocab"]
    row = 2 * 2 * kv * HEAD_DIM * case["layers"]  # bytes of K and V of one position
    n = case["prompt"]
    bytes_ = flops = 0
    if case["kind"] != "decode":  # the prompt: every weight once, its K and V written
        bytes_ += 2 * (case["layers"] * layer + head) + n * row
        flops += 2 * (n * case["layers"] * layer + head) + case["layers"] * heads * 4 * HEAD_DIM * n * (n + 1) // 2
    for i in range(case.get("steps", case.get("new", 1) - 1)):
        bytes_ += 2 * (case["layers"] * layer + head) + (n + i + 1) * row
        flops += 2 * (case["layers"] * layer + head) + case["layers"] * heads * 4 * HEAD_DIM * (n + i + 1)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """The GEMV, the decode and the default prompt form state their summation
    order and give the same bits on every path. The matrix products round an
    FP32 sum to 16 bits once (the sum's own error is far below that), and the
    prompt on the matrix cores carries its bf16 roundings through the layers."""
    if case["kind"] == "gemm":
        return {"rel": 4e-3 if case["dtype"] == "bf16" else 5e-4, "max": 2e-2 if case["dtype"] == "bf16" else 2.5e-3}
    if case.get("form") == "gemm":
        return {"rel": 2e-2, "max": 1e-1, "differ": 0.01}
    return "exact"


# ---------------------------------------------------------------- in 64 bits

def _norm(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _forward(case, seed, tokens):
    """The last position's residual row and logits, in 64 bits throughout."""
    _, _, heads, kv = SHAPES[case["shape"]]
    w = _weights(case, seed)
    n = len(tokens)
    ids = torch.from_numpy(tokens.astype(np.int64)).cuda()
    freq = THETA ** (-torch.arange(0, HEAD_DIM, 2, device="cuda", dtype=torch.float64) / HEAD_DIM)
    angle = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * freq
    cos, sin = torch.cat([angle.cos()] * 2, 1), torch.cat([angle.sin()] * 2, 1)
    causal = torch.ones((n, n), device="cuda", dtype=torch.bool).tril()

    def rope(x):
        a, b = x.chunk(2, -1)
        return x * cos + torch.cat([-b, a], -1) * sin

    x = w["model.embed_tokens.weight"][ids].double()
    for i in range(case["layers"]):
        p = {k.split(".", 3)[3][: -len(".weight")]: v.double() for k, v in w.items() if k.startswith("model.layers.%d." % i)}
        h = _norm(x, p["input_layernorm"])
        q = (h @ p["self_attn.q_proj"].T).view(n, heads, HEAD_DIM).transpose(0, 1)
        k = (h @ p["self_attn.k_proj"].T).view(n, kv, HEAD_DIM).transpose(0, 1)
        v = (h @ p["self_attn.v_proj"].T).view(n, kv, HEAD_DIM).transpose(0, 1)
        q, k = rope(_norm(q, p["self_attn.q_norm"])), rope(_norm(k, p["self_attn.k_norm"]))
        out = torch.empty((n, heads, HEAD_DIM), device="cuda", dtype=torch.float64)
        for j in range(heads):
            g = j // (heads // kv)
            s = (q[j] @ k[g].T / math.sqrt(HEAD_DIM)).masked_fill(~causal, -math.inf)
            out[:, j] = s.softmax(-1) @ v[g]
        x = x + out.reshape(n, -1) @ p["self_attn.o_proj"].T
        h = _norm(x, p["post_attention_layernorm"])
        x = x + (torch.nn.functional.silu(h @ p["mlp.gate_proj"].T) * (h @ p["mlp.up_proj"].T)) @ p["mlp.down_proj"].T
    last = x[-1]
    logits = _norm(last, w["model.norm.weight"].double()) @ w["model.embed_tokens.weight"].double().T
    return logits, last


def exact(case, seed):
    if case["kind"] in ("gemv", "gemm"):
        dtype = DTYPES[case["dtype"]][1]
        if case["kind"] == "gemv":
            a, b = _uniform((case["m"], case["lda"]), dtype, seed, 1), _uniform((case["k"],), dtype, seed, 2)
            return torch.cat([r[:, : case["k"]].double() @ b.double() for r in a.split(2048)])
        a, b = _uniform((case["m"], case["k"]), dtype, seed, 1), _uniform((case["k"], case["n"]), dtype, seed, 2)
        return a.double() @ b.double()
    if case["kind"] == "chat":  # the reply's tokens are the framework's own choice
        return None
    logits, hidden = _forward(case, seed, _tokens(case, seed))
    return {"tokens": None, "logits": logits, "hidden": hidden}
