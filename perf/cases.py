"""The measured work: whole requests through a loaded model, blocks of its layers, and the kernels
that a program can call on device buffers.

Every case goes through an entry point of the package: `HipBackend.forward` (a batch of host arrays
in, logits and pooled rows out), `HipBackend.encoder_hidden` (every position of the padded batch) or
one of the `s1k_*` calls on torch tensors. Batches are the synthetic requests of
`sys1rust_amd.workloads` (states of 16 to 8192 tokens, 1 to 10 questions each), models have the
widths of ModernBERT-large and mmBERT-base with N(0, 0.02) weights, and most of them have the three
layers of the encoder's period (one global, two local) in place of its 28 or 22, so that a case is a
block whose outputs can be held to a tolerance of its own.

`exact` is the same graph in torch float64.
"""
from __future__ import annotations

import ctypes as C
import json
import math
import zlib

import numpy as np
import torch

from sys1rust_amd import _lib, workloads
from sys1rust_amd.backend import DEFAULT_TUNING, HipBackend

SHAPES = {"large": workloads.MODERNBERT_LARGE, "base": workloads.MMBERT_BASE}
TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
STORED = {"bf16": "BF16", "f16": "F16", "f32": "F32"}
SCORER = workloads.SCORER_WIDTH
VOCAB = 50368  # ids are drawn below 50285 at every width
MASKED = -1e4  # the logit of a slot without a marker


def listed():
    model = {"shape": "large", "layers": 3, "dtype": "bf16"}
    return [
        # One question about a short state, the whole 28-layer model: a served request at its
        # smallest, where launches and latency count. f16 is what the Rust binding loads.
        {"name": "request_1q128", "kind": "forward", "shape": "large", "layers": 28, "dtype": "f16",
         "requests": 1, "questions": 1, "lo": 128, "hi": 128, "max_len": 1024},
        # Ten questions about a 512-token state, the whole model: the benchmark's request.
        {"name": "request_10q512", "kind": "forward", "shape": "large", "layers": 28, "dtype": "bf16",
         "requests": 1, "questions": 10, "lo": 512, "hi": 512, "max_len": 1024},
        # An ordinary batch of the multilingual width: two requests of three questions.
        {"name": "block_base_6rows", "kind": "forward", **model, "shape": "base", "dtype": "f16",
         "requests": 2, "questions": 3, "lo": 200, "hi": 420, "max_len": 1024},
        # 64 requests with states of 128 to 2048 tokens, three questions each: bulk scoring.
        {"name": "block_sweep64", "kind": "forward", **model,
         "requests": 64, "questions": 3, "lo": 128, "hi": 2048, "max_len": 8192},
        # One state at the model's longest: attention over 8192 keys.
        {"name": "block_8192", "kind": "forward", **model, "dtype": "f16",
         "requests": 1, "questions": 1, "lo": 8192, "hi": 8192, "max_len": 8192},
        # Hidden states of a ragged padded batch, padding positions included.
        {"name": "hidden_ragged", "kind": "hidden", **model,
         "requests": 8, "questions": 1, "lo": 40, "hi": 640, "max_len": 1024},
        # The f32 option (f32 weights and compute) for a short request and for the ten questions.
        {"name": "block_f32_1q128", "kind": "forward", **model, "dtype": "f32",
         "requests": 1, "questions": 1, "lo": 128, "hi": 128, "max_len": 1024},
        {"name": "block_f32_10q512", "kind": "forward", **model, "dtype": "f32",
         "requests": 1, "questions": 10, "lo": 512, "hi": 512, "max_len": 1024},
        # Single kernels. The MLP's first product with its GeGLU at the ten-question request, the
        # residual product of a one-question request, attention over ragged rows, a LayerNorm.
        {"name": "gemm_geglu", "kind": "gemm", "m": 5686, "n": 5248, "k": 1024, "epi": 2},
        {"name": "gemm_residual", "kind": "gemm", "m": 563, "n": 1024, "k": 2624, "epi": 1},
        {"name": "attention_rows", "kind": "attention", "rows": 12, "lo": 300, "hi": 1100, "heads": 16, "window": -1},
        {"name": "layernorm", "kind": "layernorm", "m": 5686, "d": 1024, "bias": False},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "f32", "hidden", "gemm", "attention", "layernorm"])
    shape = rng.choice(["large", "large", "base"])
    dtype = rng.choice(["bf16", "f16"])
    if kind in ("forward", "f32", "hidden"):
        requests = _spread(rng, 1, 48 if kind == "forward" else 4)
        questions = rng.randint(1, 10) if requests <= 4 else rng.randint(1, 3)
        most = {"forward": 120000, "f32": 9000, "hidden": 12000}[kind]  # rows x tokens
        hi = _spread(rng, 32, max(64, min(8000, most // (requests * questions))))
        c = {"kind": "hidden" if kind == "hidden" else "forward", "shape": shape, "layers": 3,
             "dtype": "f32" if kind == "f32" else dtype, "requests": requests, "questions": questions,
             "lo": rng.randint(max(16, hi // 4), hi), "hi": hi, "max_len": 8192}
        if kind == "hidden" and hi > 800:
            c["lo"], c["hi"] = 100, 800
        return c
    if kind == "gemm":
        n, k = rng.choice([(3072, 1024), (1024, 1024), (5248, 1024), (1024, 2624), (4096, 1024), (1024, 4096),
                           (2304, 768), (768, 768), (768, 1152)])
        epi = 2 if n == 5248 else rng.choice([0, 1, 3])
        return {"kind": "gemm", "m": _spread(rng, 1, 60000), "n": n, "k": k, "epi": epi}
    if kind == "attention":
        rows = _spread(rng, 1, 48)
        hi = _spread(rng, 16, min(8192, 40000 // rows))
        return {"kind": "attention", "rows": rows, "lo": rng.randint(1, hi), "hi": hi, "heads": rng.choice([12, 16]),
                "window": rng.choice([-1, 64])}
    return {"kind": "layernorm", "m": _spread(rng, 1, 200000), "d": rng.choice([768, 1024]),
            "bias": rng.choice([False, True])}


# ---- models: configuration, weights, batches


def _config(case):
    cfg = dict(SHAPES[case["shape"]])
    cfg.update(num_hidden_layers=case["layers"], vocab_size=VOCAB, pad_token_id=workloads.PAD)
    return cfg


def _agent(case):
    return dict(workloads.AGENT, max_len=case["max_len"])


def _weights(case, seed):
    """The checkpoint's tensors by name, on the GPU, in the type that it stores."""
    cfg = _config(case)
    d, inter, dt = cfg["hidden_size"], cfg["intermediate_size"], TORCH[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = {}

    def put(name, *shape, mean=0.0):
        x = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)
        w[name] = x.mul_(0.02).add_(mean).to(dt)

    def norm(name, bias=True):
        put(name + ".weight", d, mean=1.0)
        if bias:
            put(name + ".bias", d)

    put("encoder.embeddings.tok_embeddings.weight", VOCAB, d)
    norm("encoder.embeddings.norm", bias=False)
    for l in range(cfg["num_hidden_layers"]):
        p = f"encoder.layers.{l}"
        if l:
            norm(p + ".attn_norm", bias=False)
        put(p + ".attn.Wqkv.weight", 3 * d, d)
        put(p + ".attn.Wo.weight", d, d)
        norm(p + ".mlp_norm", bias=False)
        put(p + ".mlp.Wi.weight", 2 * inter, d)
        put(p + ".mlp.Wo.weight", d, inter)
    norm("encoder.final_norm", bias=False)
    put("type_emb.weight", 3, d)
    for j in range(_agent(case)["head_layers"]):
        p = f"head.layers.{j}"
        norm(p + ".norm1")
        put(p + ".self_attn.in_proj_weight", 3 * d, d)
        put(p + ".self_attn.in_proj_bias", 3 * d)
        put(p + ".self_attn.out_proj.weight", d, d)
        put(p + ".self_attn.out_proj.bias", d)
        norm(p + ".norm2")
        put(p + ".linear1.weight", 4 * d, d)
        put(p + ".linear1.bias", 4 * d)
        put(p + ".linear2.weight", d, 4 * d)
        put(p + ".linear2.bias", d)
    norm("scorer.0")
    put("scorer.1.weight", SCORER, d)
    put("scorer.1.bias", SCORER)
    put("scorer.3.weight", 1, SCORER)
    put("scorer.3.bias", 1, mean=1.0)  # scores around 1: around 0 their relative error says nothing
    put("act_head.0.weight", 256, d + 4)
    put("act_head.0.bias", 256)
    put("act_head.2.weight", workloads.N_ACT, 256)
    put("act_head.2.bias", workloads.N_ACT)
    return w


def _checkpoint(case, seed):
    """The safetensors image of `_weights`."""
    w = _weights(case, seed)
    header, at = {}, 0
    for name, x in w.items():
        size = x.numel() * x.element_size()
        header[name] = {"dtype": STORED[case["dtype"]], "shape": list(x.shape), "data_offsets": [at, at + size]}
        at += size
    head = json.dumps(header).encode()
    head += b" " * (-len(head) % 64)
    image = bytearray(8 + len(head) + at)
    image[:8] = len(head).to_bytes(8, "little")
    image[8: 8 + len(head)] = head
    body = torch.frombuffer(image, dtype=torch.uint8, offset=8 + len(head))
    flat = torch.cat([x.reshape(-1).view(torch.uint8) for x in w.values()])
    body.copy_(flat)
    return image


def _sizes(case):
    """Draws the lengths of a case, the same for every seed of its contents."""
    return np.random.default_rng(zlib.crc32(json.dumps({k: v for k, v in case.items() if k != "name"}).encode()))


def _batch(case, seed):
    rng, size = np.random.default_rng(seed), _sizes(case)
    agent = _agent(case)
    kinds = [("choice", 3), ("score", 4), ("noul", 2)]
    items = []
    for _ in range(case["requests"]):
        length = int(size.integers(case["lo"], case["hi"] + 1))
        questions = []
        for j in range(case["questions"]):
            kind, options = kinds[j % 3] if case["questions"] > 1 else kinds[0]
            head = rng.integers(0, workloads.RANDOM_ID_HIGH, size=int(size.integers(13, 34))).tolist()
            opts = [rng.integers(0, workloads.RANDOM_ID_HIGH, size=int(size.integers(6, 11))).tolist()
                    for _ in range(options)]
            questions.append(workloads.Question(kind, head, opts))
        items.extend(workloads.request_rows(rng, length, questions, agent["max_len"], agent["head_max_len"]))
    return workloads.collate(items)


def _settings(case):
    # The string that every served model runs with; the Rust binding puts the type before it, or
    # dtype=f32 after it.
    return f"dtype={case['dtype']},{DEFAULT_TUNING}" if case["dtype"] != "f32" else DEFAULT_TUNING + ",dtype=f32"


def _prepare_model(case, seed):
    cfg, agent = json.dumps(_config(case)), json.dumps(_agent(case))
    m = HipBackend(_checkpoint(case, seed), cfg, agent, settings=_settings(case))
    m.warmup()
    return {"kind": case["kind"], "model": m, "batch": _batch(case, seed)}


# ---- kernels on device buffers


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, scale=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).mul_(scale).to(dtype)


def _gemm_inputs(case, seed):
    m, n, k, epi = case["m"], case["n"], case["k"], case["epi"]
    gen = _gen(seed)
    s = {"a": _normal(gen, m, k), "w": _normal(gen, n, k, scale=0.02)}
    s["bias"] = None if epi == 2 else _normal(gen, n, scale=0.02, dtype=torch.float32)
    if epi == 1:  # the residual stream, added to in place
        s["c"] = _normal(gen, m, n, dtype=torch.float32)
    elif epi == 3:
        s["c"] = torch.empty(m, n, dtype=torch.float32, device="cuda")
    else:
        s["c"] = torch.empty(m, n // 2 if epi == 2 else n, dtype=torch.bfloat16, device="cuda")
    return s


def _starts(case):
    lens = _sizes(case).integers(case["lo"], case["hi"] + 1, size=case["rows"])
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def _attention_inputs(case, seed):
    starts, gen, heads = _starts(case), _gen(seed), case["heads"]
    t = int(starts[-1])
    s = {"starts": starts, "q": _normal(gen, heads, t, 64), "k": _normal(gen, heads, t, 64)}
    s["v"] = torch.zeros(heads, 64, _lib.vt_ld(t), dtype=torch.bfloat16, device="cuda")  # transposed, zeros past t
    s["v"][:, :, :t] = _normal(gen, heads, 64, t)
    s["out"] = torch.empty(t, heads * 64, dtype=torch.bfloat16, device="cuda")
    return s


def _layernorm_inputs(case, seed):
    gen, m, d = _gen(seed), case["m"], case["d"]
    s = {"x": _normal(gen, m, d, scale=3.0, dtype=torch.float32),
         "w": _normal(gen, d, scale=0.02, dtype=torch.float32) + 1.0,
         "b": _normal(gen, d, scale=0.02, dtype=torch.float32) if case["bias"] else None}
    s["y"] = torch.empty(m, d, dtype=torch.bfloat16, device="cuda")
    return s


INPUTS = {"gemm": _gemm_inputs, "attention": _attention_inputs, "layernorm": _layernorm_inputs}


def prepare(case, seed):
    if case["kind"] in ("forward", "hidden"):
        return _prepare_model(case, seed)
    return dict(INPUTS[case["kind"]](case, seed), **case)


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def run(state):
    kind, L = state["kind"], _lib.lib()
    if kind == "forward":
        out = state["model"].forward(state["batch"])
        return {"logits": out.logits, "pooled": out.pooled}
    if kind == "hidden":
        return {"hidden": state["model"].encoder_hidden(state["batch"])}
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if kind == "gemm":
        m, n, k, c = state["m"], state["n"], state["k"], state["c"]
        _lib.check(L.s1k_gemm(_ptr(state["a"]), k, _ptr(state["w"]), k, _ptr(c), c.shape[1],
                              C.cast(_ptr(state["bias"]), C.c_void_p), m, n, k, state["epi"], 0, stream))
        return c
    if kind == "attention":
        st = state["starts"]
        _lib.check(L.s1k_attention(_ptr(state["q"]), _ptr(state["k"]), _ptr(state["v"]), state["v"].shape[2],
                                   int(st[-1]), state["heads"], st.ctypes.data_as(_lib.i32p), len(st) - 1,
                                   state["window"], 0.125, _ptr(state["out"]), stream))
        return state["out"]
    _lib.check(L.s1k_layernorm(_ptr(state["x"]), _ptr(state["w"]), _ptr(state["b"]), 1e-5, state["m"], state["d"],
                               _ptr(state["y"]), stream))
    return state["y"]


# ---- the least work of a pass


def _pairs(lens, window):
    """Query-key pairs of rows of these lengths (window < 0: all of a row's)."""
    if window < 0:
        return float(sum(x * x for x in lens))
    return float(sum(x * min(x, 2 * window + 1) for x in lens))


def _model_work(case):
    cfg, b = _config(case), _batch(case, 0)
    d, inter, layers = cfg["hidden_size"], cfg["intermediate_size"], case["layers"]
    size = 4 if case["dtype"] == "f32" else 2
    lens = [float(b.len)] * b.n if case["kind"] == "hidden" else [float(x) for x in b.seq_lens]
    t, window = sum(lens), cfg["local_attention"] // 2
    per_layer = 4 * d * d + 3 * d * inter  # weights
    n_global = (layers + 2) // 3
    flops = 2.0 * t * per_layer * layers
    flops += 4.0 * d * (n_global * _pairs(lens, -1) + (layers - n_global) * _pairs(lens, window))
    weights = layers * per_layer
    if case["kind"] == "hidden":
        out = 4.0 * t * d
    else:
        # The head: its first layer over every token, of its last one only the keys and values there,
        # the rest at position 0 and the markers, and the scorer at the markers.
        picked, marked = b.n * (1 + b.kmax), b.n * b.kmax
        flops += 2.0 * t * 12 * d * d + 4.0 * d * _pairs(lens, -1)
        flops += 2.0 * t * 2 * d * d + 2.0 * picked * 10 * d * d + 4.0 * d * (1 + b.kmax) * t
        flops += 2.0 * marked * SCORER * (d + 1)
        weights += 2 * 12 * d * d + SCORER * (d + 1)
        out = 4.0 * (marked + b.n * d)
    return {"bytes": float(size) * (weights + t * d) + 8.0 * b.n * b.len + out, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("forward", "hidden"):
        return _model_work(case)
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        out = {0: 2.0, 1: 8.0, 2: 1.0, 3: 4.0}[case["epi"]]  # bytes of the result per product element
        return {"bytes": 2.0 * (m * k + n * k) + out * m * n, "flops": 2.0 * m * n * k}
    if kind == "attention":
        lens = np.diff(_starts(case)).astype(np.float64)
        return {"bytes": 8.0 * float(sum(lens)) * case["heads"] * 64,
                "flops": 4.0 * 64 * case["heads"] * _pairs(lens, case["window"])}
    return {"bytes": 6.0 * case["m"] * case["d"], "flops": 8.0 * case["m"] * case["d"]}


# ---- tolerances: four times the difference seen between two correct orders of the same sums


def tolerance(case):
    kind = case["kind"]
    if kind == "gemm":
        # f32 results differ by the order of their sums; 16-bit ones by roundings that fall the other way.
        return {"rel": 1e-5, "max": 1e-4} if case["epi"] in (1, 3) else {"rel": 1e-3, "max": 0.05}
    if kind == "attention":
        return {"rel": 5e-3, "max": 0.1}  # the softmax weights are rounded to bf16 by their running maximum
    if kind == "layernorm":
        return {"rel": 1e-3, "max": 0.02}
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 5e-4}
    if case["dtype"] == "f16":
        return {"rel": 3e-3, "max": 0.1}
    return {"rel": 2.5e-2 if case["layers"] > 6 else 1.2e-2, "max": 0.4}


# ---- the same results in 64 bits


def _ln(x, w, b=None, eps=1e-5):
    x = x - x.mean(-1, keepdim=True)
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w
    return y if b is None else y + b


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x * 0.7071067811865476))


def _rope(x, theta):
    """The half-split rotation of [heads, len, 64]; the angle is the model's, in 32 bits."""
    half = x.shape[-1] // 2
    base = np.float32(np.log2(np.float64(np.float32(theta))))
    i = np.arange(half, dtype=np.float32)
    inv = np.exp2((-(i / np.float32(half)) * base).astype(np.float64)).astype(np.float32)
    angle = np.arange(x.shape[1], dtype=np.float32)[:, None] * inv[None, :]
    a = torch.from_numpy(angle.astype(np.float64)).to(x.device)
    c, s = torch.cos(a), torch.sin(a)
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x1 * s + x2 * c], dim=-1)


def _heads(x, n):
    return x.reshape(x.shape[0], n, -1).transpose(0, 1).contiguous()


def _attend(q, k, v, scale, allow=None, count=None, zeros=None):
    """Softmax attention, a head at a time. allow [len, len]: the visible keys; count: how often each
    is counted; zeros [len]: slots of zero key and value that each query sees besides."""
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        s = (q[h] @ k[h].T) * scale
        if allow is not None:
            s = s.masked_fill(~allow, -math.inf)
        top = s.amax(-1, keepdim=True).clamp_min(0.0 if zeros is not None else -math.inf)
        e = torch.exp(s - top)
        if count is not None:
            e = e * count
        total = e.sum(-1, keepdim=True)
        if zeros is not None:
            total = total + zeros[:, None] * torch.exp(-top)
        out[h] = (e @ v[h]) / total
    return out.transpose(0, 1).reshape(q.shape[1], -1)


def _padded_keys(length, real, window):
    """The keys of each position of a padded row of `length` with `real` tokens on a local layer, under
    the settings of `_settings`: (allow, zero slots). A padding position with a real key in its window
    sees those; a farther one sees its window and every real key (rows up to 511), or the real keys of
    its chunk and its window, positions past the row as zero slots (the banded form, from 512)."""
    i = torch.arange(length, device="cuda")
    near = (i[:, None] - i[None, :]).abs() <= window
    is_real = (i < real)[None, :]
    allow, zeros = near & is_real, torch.zeros(length, dtype=torch.float64, device="cuda")
    far = i >= real + window
    if bool(far.any()):
        seen = is_real.expand(length, length)
        if length >= 512:
            chunk = i // window
            seen = seen & (i[None, :] >= ((chunk - 1) * window)[:, None])
            past = (i + window + 1 - length).clamp_min(0).to(torch.float64)
            zeros = torch.where(far, past, zeros)
        allow = torch.where(far[:, None], near | seen, allow)
    return allow, zeros


def _exact_encoder(cfg, w, ids, real):
    d, nh, inter, eps = cfg["hidden_size"], cfg["num_attention_heads"], cfg["intermediate_size"], cfg["norm_eps"]
    length, window = len(ids), cfg["local_attention"] // 2
    theta = {g: cfg["rope_parameters"][k]["rope_theta"] for g, k in ((True, "full_attention"), (False, "sliding_attention"))}
    idt = torch.from_numpy(ids.astype(np.int64)).cuda()
    h = _ln(w["encoder.embeddings.tok_embeddings.weight"][idt].double(), w["encoder.embeddings.norm.weight"], None, eps)
    i = torch.arange(length, device="cuda")
    for l in range(cfg["num_hidden_layers"]):
        p, full = f"encoder.layers.{l}", l % cfg["global_attn_every_n_layers"] == 0
        x = _ln(h, w[p + ".attn_norm.weight"], None, eps) if l else h
        q, k, v = (_heads(y, nh) for y in (x @ w[p + ".attn.Wqkv.weight"].T).split(d, dim=-1))
        q, k = _rope(q, theta[full]), _rope(k, theta[full])
        if full:
            att = _attend(q, k, v, 0.125, None if real == length else (i < real)[None, :].expand(length, length))
        elif real == length and length > 2000:  # a long row's window, a stretch of queries at a time
            att = torch.empty(length, d, dtype=torch.float64, device="cuda")
            for a in range(0, length, 1024):
                e, lo, hi = min(length, a + 1024), max(0, a - window), min(length, a + 1024 + window)
                near = (i[a:e, None] - i[None, lo:hi]).abs() <= window
                for g in range(nh):
                    s = ((q[g, a:e] @ k[g, lo:hi].T) * 0.125).masked_fill(~near, -math.inf)
                    att[a:e, g * 64: g * 64 + 64] = torch.softmax(s, -1) @ v[g, lo:hi]
        else:
            allow, zeros = _padded_keys(length, real, window)
            att = _attend(q, k, v, 0.125, allow, None, zeros if bool(zeros.any()) else None)
        h = h + att @ w[p + ".attn.Wo.weight"].T
        x, g = (_ln(h, w[p + ".mlp_norm.weight"], None, eps) @ w[p + ".mlp.Wi.weight"].T).split(inter, dim=-1)
        h = h + (_gelu(x) * g) @ w[p + ".mlp.Wo.weight"].T
    return _ln(h, w["encoder.final_norm.weight"], None, eps)


def _exact_head(cfg, agent, w, h, picked):
    d, nh = cfg["hidden_size"], cfg["num_attention_heads"]
    for j in range(agent["head_layers"]):
        p = f"head.layers.{j}"
        x = _ln(h, w[p + ".norm1.weight"], w[p + ".norm1.bias"])
        qkv = x @ w[p + ".self_attn.in_proj_weight"].T + w[p + ".self_attn.in_proj_bias"]
        q, k, v = (_heads(y, nh) for y in qkv.split(d, dim=-1))
        if j + 1 == agent["head_layers"]:
            h, q = h[picked], q[:, picked]
        h = h + _attend(q, k, v, 0.125) @ w[p + ".self_attn.out_proj.weight"].T + w[p + ".self_attn.out_proj.bias"]
        x = _ln(h, w[p + ".norm2.weight"], w[p + ".norm2.bias"])
        x = torch.relu(x @ w[p + ".linear1.weight"].T + w[p + ".linear1.bias"])
        h = h + x @ w[p + ".linear2.weight"].T + w[p + ".linear2.bias"]
    s = _ln(h[1:], w["scorer.0.weight"], w["scorer.0.bias"])
    s = _gelu(s @ w["scorer.1.weight"].T + w["scorer.1.bias"])
    return (s @ w["scorer.3.weight"].T + w["scorer.3.bias"]).reshape(-1), h[0]


def _exact_model(case, seed):
    cfg, agent, b = _config(case), _agent(case), _batch(case, seed)
    w = {k: x if "tok_embeddings" in k else x.double() for k, x in _weights(case, seed).items()}
    ids = b.input_ids.reshape(b.n, b.len)
    if case["kind"] == "hidden":
        rows = [_exact_encoder(cfg, w, ids[r], int(b.seq_lens[r])) for r in range(b.n)]
        return {"hidden": torch.stack(rows).reshape(-1)}
    logits = np.full((b.n, b.kmax), MASKED, dtype=np.float64)
    pooled = []
    for r in range(b.n):
        real, live = int(b.seq_lens[r]), int(b.marker_count[r])
        h = _exact_encoder(cfg, w, ids[r, :real], real) + w["type_emb.weight"][int(b.qtype[r])]
        markers = b.marker_pos.reshape(b.n, b.kmax)[r, :live].astype(np.int64).tolist()
        lg, top = _exact_head(cfg, agent, w, h, [0] + markers)
        logits[r, :live] = lg.cpu().numpy()
        pooled.append(top)
    return {"logits": logits.reshape(-1), "pooled": torch.cat(pooled)}


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "hidden"):
        return _exact_model(case, seed)
    s = INPUTS[kind](case, seed)
    if kind == "gemm":
        c = s["a"].double() @ s["w"].double().T
        if case["epi"] == 2:  # weight rows come in blocks of 32: the product, then its gate
            c = c.reshape(case["m"], -1, 2, 32)
            return (_gelu(c[:, :, 0]) * c[:, :, 1]).reshape(case["m"], -1)
        c = c + s["bias"].double()
        return c + s["c"].double() if case["epi"] == 1 else c
    if kind == "attention":
        out, st = [], s["starts"]
        q, k, v = (x.double() for x in (s["q"], s["k"], s["v"].transpose(1, 2)))
        for a, e in zip(st[:-1].tolist(), st[1:].tolist()):
            i = torch.arange(e - a, device="cuda")
            allow = None if case["window"] < 0 else (i[:, None] - i[None, :]).abs() <= case["window"]
            out.append(_attend(q[:, a:e], k[:, a:e], v[:, a:e], 0.125, allow))
        return torch.cat(out)
    return _ln(s["x"].double(), s["w"].double(), None if s["b"] is None else s["b"].double())
