"""The token loop's work as a user of this framework meets it, as cases to be timed and compared.

Whole calls of the step API (decode steps, a speculative verify batch, prefill) run on models of this
repository's own shapes, with random weights: the 0.6B shape in full, the larger ones with a few of their
layers. The rest are single layers' work through the kernel entry points: quantized projections at one
token (decode), a few tokens (verify) and many (prefill), and prefill attention.

Weights are uniform code words whose scale and bias centre them on zero with a spread of 0.02, like a
trained projection's; activations are N(0, 1) in fp32, as the RMSNorms leave them. Projections of one or a
few tokens run over a stack of matrices (one pass reads each once), so that they come from memory and not
from a cache, as in a model's token loop.
"""
import ctypes
import json
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mlx-runner_amd"))

import configs  # noqa: E402
import mlxr  # noqa: E402

GREEDY = mlxr.SamplingParameters.greedy()
D = 128            # head_dim of every supported model
PAGE = 64          # positions per KV-cache page
STACK = 320 << 20  # bytes of weights one pass of a matrix stack reads, about (at least one matrix)


# ------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest model in full, a short chat turn: 8 tokens after 96, launches and hand-overs count
        {"name": "decode-0.6b", "kind": "decode", "model": "qwen3-0.6b", "layers": 28, "bits": 4, "gs": 64, "context": 96, "steps": 8},
        # 8B layers and head at a usual chat context
        {"name": "decode-8b-4k", "kind": "decode", "model": "qwen3-8b", "layers": 4, "bits": 4, "gs": 64, "context": 4090, "steps": 8},
        # long context with the sparse decode attention: 32B layers, 24 thousand tokens
        {"name": "decode-32b-sparse-24k", "kind": "decode", "model": "qwen2.5-32b", "layers": 4, "bits": 4, "gs": 64, "context": 24001,
         "steps": 4, "sparse": True},
        # a drafted continuation of four tokens checked in one pass, logits of every row
        {"name": "verify-8b-t5", "kind": "verify", "model": "qwen3-8b", "layers": 4, "bits": 4, "gs": 64, "context": 4090, "tokens": 5},
        # a prompt of one full chunk
        {"name": "prefill-8b-2048", "kind": "prefill", "model": "llama3-8b", "layers": 4, "bits": 4, "gs": 64, "context": 0, "tokens": 2048},
        # a second turn: a ragged prompt after a reused prefix
        {"name": "prefill-8b-300-at-1500", "kind": "prefill", "model": "llama3-8b", "layers": 4, "bits": 4, "gs": 64, "context": 1500, "tokens": 300},
        # projections of models that are not 4-bit, one decode token each: a down projection ...
        {"name": "matvec-q6-14336-4096", "kind": "linear", "tokens": 1, "K": 14336, "O": 4096, "bits": 6, "gs": 128},
        # ... and the 8-bit lm_head
        {"name": "matvec-q8-4096-151936", "kind": "linear", "tokens": 1, "K": 4096, "O": 151936, "bits": 8, "gs": 64},
        # the same models' verify batch
        {"name": "batch4-q8-4096-14336", "kind": "linear", "tokens": 4, "K": 4096, "O": 14336, "bits": 8, "gs": 64},
        # and their prefill: one of the reference's 512-token chunks, and a short ragged prompt
        {"name": "gemm512-q8-4096-14336", "kind": "linear", "tokens": 512, "K": 4096, "O": 14336, "bits": 8, "gs": 64},
        {"name": "gemm77-q3-14336-4096", "kind": "linear", "tokens": 77, "K": 14336, "O": 4096, "bits": 3, "gs": 32},
        # one layer's attention over a later chunk of a long prompt, at the 32B head shape
        {"name": "flash-1000-at-7001", "kind": "flash", "tokens": 1000, "context": 7001, "heads": 40, "kv_heads": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "verify", "prefill", "matvec", "matvec", "batch", "batch", "gemm", "gemm", "flash"])
    if kind == "decode":
        if rng.random() < 0.25:
            return {"kind": kind, "model": "qwen2.5-32b", "layers": 4, "bits": 4, "gs": 64, "context": _log(rng, 6000, 24000),
                    "steps": rng.randint(1, 4), "sparse": True}
        name, layers = rng.choice([("qwen3-0.6b", 28), ("qwen3-8b", 4)])
        return {"kind": kind, "model": name, "layers": layers, "bits": 4, "gs": 64, "context": _log(rng, 12, 8000), "steps": rng.randint(1, 8)}
    if kind == "verify":
        return {"kind": kind, "model": "qwen3-8b", "layers": 4, "bits": 4, "gs": 64, "context": _log(rng, 30, 8000), "tokens": rng.randint(2, 8)}
    if kind == "prefill":
        return {"kind": kind, "model": "llama3-8b", "layers": 4, "bits": 4, "gs": 64, "context": rng.choice([0, _log(rng, 20, 3000)]),
                "tokens": _log(rng, 9, 2048)}
    if kind == "flash":
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "tokens": _log(rng, 16, 1000), "context": rng.choice([0, _log(rng, 50, 7000)]), "heads": kv * rng.choice([1, 2, 4, 5]),
                "kv_heads": kv}
    bits, gs = rng.choice([(3, 32), (3, 64), (4, 64), (6, 64), (6, 128), (8, 32), (8, 64)])
    K = 128 * _log(rng, 1024 // 128, 14336 // 128)
    O = _log(rng, 500, 30000)
    T = 1 if kind == "matvec" else rng.randint(2, 8) if kind == "batch" else _log(rng, 9, 512)
    return {"kind": "linear", "tokens": T, "K": K, "O": O, "bits": bits, "gs": gs}


# ------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _matrix(gen, O, K, bits, gs):
    """Code words [O][K bits / 32] (int32), scales and biases [O][K / gs] (bf16) of a random matrix."""
    w = torch.randint(-2**31, 2**31, (O, K * bits // 32), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    top = 2**bits - 1
    s = (torch.rand((O, K // gs), generator=gen, device="cuda") + 0.5) * (0.02 * math.sqrt(12) / top)
    s = s.to(torch.bfloat16)
    b = (s.float() * (-0.5 * top)).to(torch.bfloat16)
    return w, s, b


def _config(case):
    cfg = configs.with_layers(configs.CONFIGS[case["model"]], case["layers"])
    cfg["quantization"] = {"bits": case["bits"], "group_size": case["gs"]}
    return cfg


def _tensors(cfg):
    """(name, kind, rows, columns) of a model's tensors: quantized matrices, norm weights (ones), bias rows."""
    H, I = cfg["hidden_size"], cfg["intermediate_size"]
    nH, nKV, V = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["vocab_size"]
    yield "model.embed_tokens", "matrix", V, H
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        for n, rows in (("q", nH * D), ("k", nKV * D), ("v", nKV * D)):
            yield p + f"self_attn.{n}_proj", "matrix", rows, H
            if cfg["model_type"] == "qwen2":
                yield p + f"self_attn.{n}_proj.bias", "bias", rows, 0
        yield p + "self_attn.o_proj", "matrix", H, nH * D
        yield p + "mlp.gate_proj", "matrix", I, H
        yield p + "mlp.up_proj", "matrix", I, H
        yield p + "mlp.down_proj", "matrix", H, I
        yield p + "input_layernorm.weight", "norm", H, 0
        yield p + "post_attention_layernorm.weight", "norm", H, 0
        if cfg["model_type"] == "qwen3":
            yield p + "self_attn.q_norm.weight", "norm", D, 0
            yield p + "self_attn.k_norm.weight", "norm", D, 0
    yield "model.norm.weight", "norm", H, 0
    if not cfg["tie_word_embeddings"]:
        yield "lm_head", "matrix", V, H


def _model_dir(cfg):
    """The model's directory (config.json, model.safetensors), written on first use."""
    q = cfg["quantization"]
    name = "{}-{}l-q{}g{}".format(cfg["model_type"] + str(cfg["hidden_size"]), cfg["num_hidden_layers"], q["bits"], q["group_size"])
    base = os.path.join(tempfile.gettempdir(), f"mlxr_perf_{os.getuid()}")
    path = os.path.join(base, name)
    if os.path.exists(path):
        return path
    os.makedirs(base, exist_ok=True)
    tmp = tempfile.mkdtemp(dir=base)
    gen, header, offset, order = _generator(17), {}, 0, []
    for name, kind, rows, cols in _tensors(cfg):
        if kind == "matrix":
            parts = [(name + ".weight", "U32", [rows, cols * q["bits"] // 32], 4),
                     (name + ".scales", "BF16", [rows, cols // q["group_size"]], 2),
                     (name + ".biases", "BF16", [rows, cols // q["group_size"]], 2)]
        else:
            parts = [(name, "BF16", [rows], 2)]
        for key, dtype, shape, size in parts:
            n = int(np.prod(shape)) * size
            header[key] = {"dtype": dtype, "shape": shape, "data_offsets": [offset, offset + n]}
            offset += n
        order.append((kind, rows, cols))
    text = json.dumps(header)
    text += " " * (-(8 + len(text)) % 8)
    with open(os.path.join(tmp, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text.encode())
        for kind, rows, cols in order:
            if kind == "matrix":
                out = _matrix(gen, rows, cols, q["bits"], q["group_size"])
            elif kind == "bias":
                out = [(torch.randn(rows, generator=gen, device="cuda") * 0.02).to(torch.bfloat16)]
            else:
                out = [torch.ones(rows, device="cuda", dtype=torch.bfloat16)]
            for t in out:
                f.write(t.view(torch.uint8).cpu().numpy().tobytes())
    with open(os.path.join(tmp, "config.json"), "w") as f:
        json.dump(cfg, f)
    try:
        os.rename(tmp, path)
    except OSError:   # another process was first
        pass
    return path


def _tokens(case, seed, vocab):
    n = case["context"] + case.get("steps", case.get("tokens", 0))
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        gen = _generator(seed)
        T, K, O, bits, gs = (case[k] for k in ("tokens", "K", "O", "bits", "gs"))
        count = _count(case)
        mats = [_matrix(gen, O, K, bits, gs) for _ in range(count)]
        x = torch.randn((count, T, K), generator=gen, device="cuda")
        y = torch.zeros((count, T, O), device="cuda")
        qm = [(mlxr.QMat * 1)(mlxr.QMat(w.data_ptr(), s.data_ptr(), b.data_ptr(), None, O)) for w, s, b in mats]
        torch.cuda.synchronize()
        return {"kind": kind, "case": case, "mats": mats, "qm": qm, "x": x, "y": y}
    if kind == "flash":
        gen = _generator(seed)
        T, nH, nKV = case["tokens"], case["heads"], case["kv_heads"]
        keys = case["context"] + T
        seq = -(-keys // PAGE) * PAGE
        # cache layout: [pages][KV heads][64][128] bf16; q and k of rotated, normalised size
        k = torch.randn((seq // PAGE, nKV, PAGE, D), generator=gen, device="cuda").to(torch.bfloat16)
        v = torch.randn((seq // PAGE, nKV, PAGE, D), generator=gen, device="cuda").to(torch.bfloat16)
        q = torch.randn((T, nH * D), generator=gen, device="cuda")
        out = torch.zeros((T, nH * D), device="cuda")
        torch.cuda.synchronize()
        return {"kind": kind, "case": case, "q": q, "k": k, "v": v, "seq": seq, "out": out}
    cfg = _config(case)
    tokens = _tokens(case, seed, cfg["vocab_size"])
    sparse = mlxr.SparseAttention() if case.get("sparse") else None
    model = mlxr.Transformer(_model_dir(cfg), context_length=len(tokens) + 16, sparse=sparse)
    if case["context"]:
        model.prefill(tokens[:case["context"]], 0, GREEDY)
    logits = np.zeros((case["tokens"] if kind == "verify" else 1, model.vocab_size), np.float32)
    return {"kind": kind, "case": case, "model": model, "tokens": tokens, "logits": logits}


# -------------------------------------------------------------------------------------------- runs
def _forward(state, tokens, offset, all_logits):
    """The C entry point mlxr_forward; its logits are the model's until the next call, so they are taken
    into the program's own buffer."""
    model, out = state["model"], ctypes.POINTER(ctypes.c_float)()
    mlxr.check(mlxr.lib.mlxr_forward(model._h, tokens.ctypes.data, len(tokens), offset, int(all_logits), 0, ctypes.byref(out), mlxr.CancelFn(), None))
    np.copyto(state["logits"], np.ctypeslib.as_array(out, shape=state["logits"].shape))
    return state["logits"]


def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "linear":
        T, K, O, bits, gs = (case[k] for k in ("tokens", "K", "O", "bits", "gs"))
        x, y = state["x"], state["y"]
        for i, qm in enumerate(state["qm"]):
            xp, yp = x.data_ptr() + i * T * K * 4, y.data_ptr() + i * T * O * 4
            if T == 1:
                rc = mlxr.lib.mlxr_k_qmv(qm, 1, K, bits, gs, 0, xp, None, 0.0, yp, 0)
            elif T <= 8:
                rc = mlxr.lib.mlxr_k_qmm(qm, 1, K, bits, gs, 0, T, xp, K, yp, O)
            else:
                rc = mlxr.lib.mlxr_k_qgemm(qm, K, bits, gs, 0, T, xp, K, yp, O)
            mlxr.check(rc)
        return y
    if kind == "flash":
        nH, nKV = case["heads"], case["kv_heads"]
        mlxr.check(mlxr.lib.mlxr_k_flash_prefill(state["q"].data_ptr(), nH * D, state["k"].data_ptr(), state["v"].data_ptr(), state["seq"], D,
                                                 nH, nKV, case["context"], case["tokens"], 1 / math.sqrt(D), state["out"].data_ptr(), nH * D))
        return state["out"]
    model, tokens, at = state["model"], state["tokens"], case["context"]
    if kind == "decode":
        # the given tokens one step each (their selection on the GPU and its read-back are part of a step)
        for i in range(case["steps"]):
            model.finish(model.begin_steps(tokens[at + i:at + i + 1], at + i, GREEDY))
        return model.step_logits()
    return _forward(state, tokens[at:], at, kind == "verify")


# ------------------------------------------------------------------------------------ work, limits
def _matrix_bytes(O, K, bits, gs):
    return O * K * bits // 8 + 4 * O * (K // gs)


def _count(case):
    if case["tokens"] > 8:
        return 1
    return max(1, min(64, STACK // _matrix_bytes(case["O"], case["K"], case["bits"], case["gs"])))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        T, K, O = case["tokens"], case["K"], case["O"]
        n = _count(case)
        return {"bytes": n * (_matrix_bytes(O, K, case["bits"], case["gs"]) + 4 * T * (K + O)), "flops": n * 2 * T * K * O}
    T, c = case.get("tokens", 1), case["context"]
    if kind == "flash":
        nH, nKV = case["heads"], case["kv_heads"]
        pairs = T * c + T * (T + 1) // 2
        return {"bytes": 2 * 2 * nKV * D * (c + T) + 2 * 4 * T * nH * D, "flops": 4 * D * nH * pairs}
    cfg = _config(case)
    H, I, L, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["num_hidden_layers"], cfg["vocab_size"]
    nH, nKV = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    layer = H * (nH + 2 * nKV) * D + nH * D * H + 3 * H * I
    weight = lambda n: n * case["bits"] / 8 + 4 * n / case["gs"]  # noqa: E731
    rows = T if kind == "verify" else 1
    passes = case.get("steps", 1)
    keys = c + T
    if case.get("sparse"):   # the block index, and the attended keys: sinks, 512 blocks of 4, the window
        kv = ((keys - 512) // 4) * nKV * D * 2 + (4 + 2048 + 512) * nKV * D * 4
        keys = 4 + 2048 + 512
    else:
        kv = keys * nKV * D * 4
    pairs = T * keys - T * (T - 1) // 2
    flops = L * (2 * T * layer + 4 * D * nH * pairs) + 2 * rows * H * V
    return {"bytes": passes * (L * (weight(layer) + kv) + weight(H * V) + 4 * rows * V), "flops": passes * flops}


def tolerance(case):
    """About four times the distance from 64-bit results that the path showed when these were written."""
    if case["kind"] == "linear":
        if case["tokens"] == 1:
            return {"rel": 2e-6}     # fp32 products and sums
        # x as two f16 parts against codes in f16: the matrix cores' alignment of small codes sets the error
        return {"rel": 3e-4 if case["bits"] == 3 else 1e-4 if case["bits"] == 4 else 1e-5}
    if case["kind"] == "flash":
        return {"rel": 3e-5}         # q and the probabilities as bf16 pairs
    return {"rel": 1e-2}             # bf16 K/V cache, f16 activations in the prefill's projections


# -------------------------------------------------------------------------------------- references
def _dequant(w, s, b, bits, gs, r0, r1):
    """Rows [r0, r1) of a quantized matrix in 64 bits."""
    K = w.shape[1] * 32 // bits
    words = w[r0:r1].to(torch.int64) & 0xFFFFFFFF
    words = torch.cat([words, torch.zeros_like(words[:, :1])], 1)
    bit = torch.arange(K, device=w.device) * bits
    q = ((words[:, bit // 32] | (words[:, bit // 32 + 1] << 32)) >> (bit % 32)) & (2**bits - 1) if bits not in (4, 8) else \
        (words[:, bit // 32] >> (bit % 32)) & (2**bits - 1)
    g = lambda t: t[r0:r1].double().repeat_interleave(gs, 1)  # noqa: E731
    return q.double() * g(s) + g(b)


def _linear(x, w, s, b, bits, gs):
    rows = max(1, (1 << 25) // x.shape[1])
    return torch.cat([x @ _dequant(w, s, b, bits, gs, r, r + rows).T for r in range(0, w.shape[0], rows)], 1)


def _attention(q, k, v, at):
    """Causal attention of queries [T][heads][D] at positions at.. over keys [n][kv heads][D]."""
    T, nH, _ = q.shape
    G = nH // k.shape[1]
    out = torch.empty_like(q)
    step = max(1, (1 << 26) // k.shape[0])
    for h in range(nH):
        for t0 in range(0, T, step):
            t1 = min(T, t0 + step)
            s = (q[t0:t1, h] @ k[:, h // G].T) / math.sqrt(D)
            pos = torch.arange(at + t0, at + t1, device=q.device)
            s.masked_fill_(torch.arange(k.shape[0], device=q.device)[None] > pos[:, None], -math.inf)
            out[t0:t1, h] = torch.softmax(s, 1) @ v[:, h // G]
    return out


def _read(path):
    with open(os.path.join(path, "model.safetensors"), "rb") as f:
        n = struct.unpack("<Q", f.read(8))[0]
        header = json.loads(f.read(n))
    data = np.memmap(os.path.join(path, "model.safetensors"), np.uint8, "r", 8 + n)
    kinds = {"U32": torch.int32, "BF16": torch.bfloat16}

    def get(name):
        e = header[name]
        a, b = e["data_offsets"]
        return torch.from_numpy(np.array(data[a:b])).cuda().view(kinds[e["dtype"]]).view(e["shape"])
    return header, get


def _model_logits(case, seed):
    """Logits after the case's tokens, in 64 bits over a bf16 K/V cache (the cache's own type)."""
    cfg = _config(case)
    ids = torch.from_numpy(_tokens(case, seed, cfg["vocab_size"])).long().cuda()
    header, get = _read(_model_dir(cfg))
    bits, gs, eps = case["bits"], case["gs"], cfg["rms_norm_eps"]
    nH, nKV = cfg["num_attention_heads"], cfg["num_key_value_heads"]

    def norm(x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * get(name).double()

    def lin(x, name):
        y = _linear(x, get(name + ".weight"), get(name + ".scales"), get(name + ".biases"), bits, gs)
        return y + get(name + ".bias").double() if name + ".bias" in header else y

    n = len(ids)
    freq = 1.0 / cfg["rope_theta"] ** (torch.arange(0, D, 2, device="cuda").double() / D)
    angle = torch.arange(n, device="cuda").double()[:, None] * freq[None]
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    emb = "model.embed_tokens"
    h = _dequant(get(emb + ".weight")[ids], get(emb + ".scales")[ids], get(emb + ".biases")[ids], bits, gs, 0, n)
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        x = norm(h, p + "input_layernorm.weight")
        q, k, v = (lin(x, p + f"self_attn.{c}_proj").view(n, -1, D) for c in "qkv")
        if p + "self_attn.q_norm.weight" in header:
            q, k = norm(q, p + "self_attn.q_norm.weight"), norm(k, p + "self_attn.k_norm.weight")
        k, v = rope(k).to(torch.bfloat16).double(), v.to(torch.bfloat16).double()
        h = h + lin(_attention(rope(q), k, v, 0).view(n, nH * D), p + "self_attn.o_proj")
        x = norm(h, p + "post_attention_layernorm.weight")
        h = h + lin(torch.nn.functional.silu(lin(x, p + "mlp.gate_proj")) * lin(x, p + "mlp.up_proj"), p + "mlp.down_proj")
    rows = case["tokens"] if case["kind"] == "verify" else 1
    return lin(norm(h[-rows:], "model.norm.weight"), emb if cfg["tie_word_embeddings"] else "lm_head")


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        st = prepare(case, seed)
        return torch.stack([_linear(st["x"][i].double(), w, s, b, case["bits"], case["gs"]) for i, (w, s, b) in enumerate(st["mats"])])
    if kind == "flash":
        st = prepare(case, seed)
        keys = case["context"] + case["tokens"]
        flat = lambda t: t.transpose(1, 2).reshape(-1, case["kv_heads"], D)[:keys].double()  # noqa: E731
        q = st["q"].view(case["tokens"], case["heads"], D).double()
        return _attention(q, flat(st["k"]), flat(st["v"]), case["context"]).view(case["tokens"], -1)
    if case.get("sparse"):   # the keys a step attends are chosen by rank: near ties have no exact answer
        return None
    y = _model_logits(case, seed).cpu().numpy()
    return y[0] if kind == "decode" else y
