"""What is timed when a change to the decode engine is judged: calls through the public entry
points (Engine, Gpu) at the sizes of the Qwen3 shapes that bench.py and the tests run.

Kinds:
  linear     Gpu.gemv, the projection of n rows (Gpu::gemm): decode at n = 1, a batched step or a
             short prompt up to 64 rows, prefill past that
  mlp        Gpu.gemv_fused, the decode step's add + RMSNorm, gate/up projection and SwiGLU
  attention  Gpu.attention_split, decode attention of one token over a paged K/V cache
  stack      Engine.greedy_with_last_logits, a prompt through two layers, every row of the first
             one feeding the second one's attention
  chat       Engine.greedy_with_last_logits at full depth: prompt, then greedy tokens
  batch      Engine.greedy_batch at full depth: independent prompts decoded together
"""
import functools
import json
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "x0ne-engine_amd"))

from x0ne_core import Engine, EngineOptions, Gpu, split_state_bytes  # noqa: E402

HEAD = 128
PAGE = 16
EPS = 1e-6
THETA = 1e6
VOCAB = 151936
STACK_VOCAB = 4096
NORM, SWIGLU = 1, 2  # x0ne_gpu_gemv_fused: the norm prologue, the SwiGLU epilogue

# The Qwen3 dense shapes of bench.py.
MODELS = {
    "0.6b": dict(hidden=1024, inter=3072, layers=28, q_heads=16, kv_heads=8, tied=True, batch_std=0.0005),
    "8b": dict(hidden=4096, inter=12288, layers=36, q_heads=32, kv_heads=8, tied=False, batch_std=0.001),
    "32b": dict(hidden=5120, inter=25600, layers=64, q_heads=64, kv_heads=8, tied=False, batch_std=0.001),
}


def projections(model):
    """(rows, cols) of a layer's four projections."""
    m = MODELS[model]
    q, kv = m["q_heads"] * HEAD, m["kv_heads"] * HEAD
    return {"qkv": (q + 2 * kv, m["hidden"]), "o": (m["hidden"], q), "gate_up": (2 * m["inter"], m["hidden"]),
            "down": (m["hidden"], m["inter"])}


def linear(model, name, n, layers, f32=False):
    rows, cols = projections(model)[name]
    return {"kind": "linear", "rows": rows, "cols": cols, "n": n, "layers": layers, "f32": f32}


def attention(model, ctx, layers):
    m = MODELS[model]
    return {"kind": "attention", "q_heads": m["q_heads"], "kv_heads": m["kv_heads"], "ctx": ctx, "layers": layers}


def listed():
    return [
        # One decode step's QKV projections at the smallest model: 4096 x 1024 by one row, all 28
        # layers' launches in one graph. The smallest kernels, where launch and start-up time count.
        dict(linear("0.6b", "qkv", 1, 28), name="decode_qkv_0.6b"),
        # Half of the decode step's bytes: the fused gate/up GEMV of the 8B shape in the default
        # (exact) accumulation, four layers' weights.
        {"name": "decode_mlp_8b", "kind": "mlp", "hidden": 4096, "inter": 12288, "layers": 4, "exact_sums": True},
        # Decode attention of the 8B shape with a long conversation in the cache.
        dict(attention("8b", 8192, 8), name="decode_attention_8k"),
        # A batched decode step's largest projection: 16 rows at the 32B shape.
        dict(linear("32b", "gate_up", 16, 2), name="batch_gate_up_32b"),
        # An ordinary prompt: 200 rows (no multiple of a tile) through the 8B down projection.
        dict(linear("8b", "down", 200, 1), name="prompt_down_8b"),
        # A prefill pass's largest projection: 2048 rows, 8B gate/up.
        dict(linear("8b", "gate_up", 2048, 1), name="prefill_gate_up_8b"),
        # An ordinary prompt in the default (exact) accumulation.
        {"name": "prompt_333_exact_8b", "kind": "stack", "model": "8b", "prompt": 333, "exact_sums": True},
        # A document as prompt: four passes of 2048 rows with f32 sums.
        {"name": "prompt_8192_f32_8b", "kind": "stack", "model": "8b", "prompt": 8192, "exact_sums": False},
        # An ordinary, odd prompt at the smallest model with f32 sums.
        {"name": "prompt_777_f32_0.6b", "kind": "stack", "model": "0.6b", "prompt": 777, "exact_sums": False},
        # A short question answered by the smallest model: latency per token.
        {"name": "chat_0.6b", "kind": "chat", "model": "0.6b", "prompt": 20, "tokens": 64},
        # The same at the 8B shape (the default bench workload's step): bandwidth per token.
        {"name": "chat_8b", "kind": "chat", "model": "8b", "prompt": 20, "tokens": 64},
        # Serving: eight prompts of 512 tokens answered together.
        {"name": "batch8_8b", "kind": "batch", "model": "8b", "batch": 8, "prompt": 512, "tokens": 32},
    ]


def log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "attention", "attention", "stack", "stack", "chat", "batch"])
    if kind == "linear":
        n = log_uniform(rng, 1, 2048)
        return linear(rng.choice(["0.6b", "8b", "32b"]) if n <= 64 else rng.choice(["0.6b", "8b"]),
                      rng.choice(["qkv", "o", "gate_up", "down"]), n, 4 if n <= 64 else 1, rng.random() < 0.25)
    if kind == "mlp":
        m = MODELS[rng.choice(["0.6b", "8b", "32b"])]
        return {"kind": "mlp", "hidden": m["hidden"], "inter": m["inter"], "layers": rng.choice([2, 3, 4]),
                "exact_sums": rng.random() < 0.7}
    if kind == "attention":
        return attention(rng.choice(["0.6b", "8b", "32b"]), log_uniform(rng, 16, 32768), 4)
    if kind == "stack":
        exact_sums = rng.random() < 0.5
        return {"kind": "stack", "model": rng.choice(["0.6b", "8b"]),
                "prompt": log_uniform(rng, 8, 1024 if exact_sums else 8192), "exact_sums": exact_sums}
    if kind == "chat":
        return {"kind": "chat", "model": "0.6b", "prompt": log_uniform(rng, 4, 512), "tokens": rng.randint(16, 64)}
    return {"kind": "batch", "model": rng.choice(["0.6b", "8b"]), "batch": rng.randint(2, 8),
            "prompt": log_uniform(rng, 16, 512), "tokens": rng.randint(4, 32)}


# -- inputs --

@functools.lru_cache(maxsize=None)
def gpu():
    """The program's one device handle."""
    return Gpu()


def normal(g, shape, std):
    """N(0, std) in bf16, drawn on the GPU."""
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, std, generator=g)


def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def config(model, layers, vocab, tied):
    m = MODELS[model]
    return {"model_type": "qwen3", "dtype": "bfloat16", "hidden_act": "silu", "attention_bias": False,
            "hidden_size": m["hidden"], "intermediate_size": m["inter"], "num_hidden_layers": layers,
            "num_attention_heads": m["q_heads"], "num_key_value_heads": m["kv_heads"], "head_dim": HEAD,
            "vocab_size": vocab, "max_position_embeddings": 40960, "rms_norm_eps": EPS, "rope_theta": THETA,
            "tie_word_embeddings": tied}


def linear_inputs(case, seed):
    """Weights N(0, 0.02), rows N(0, 1) (they come out of a norm)."""
    g = generator(seed)
    return [(normal(g, (case["rows"], case["cols"]), 0.02), normal(g, (case["n"], case["cols"]), 1.0))
            for _ in range(case["layers"])]


def mlp_inputs(case, seed):
    g, h = generator(seed), case["hidden"]
    return [{"w": normal(g, (2 * case["inter"], h), 0.02), "delta": normal(g, (h,), 0.3),
             "res_in": torch.empty(h, device="cuda").normal_(0.0, 1.0, generator=g),
             "norm_w": (1.0 + normal(g, (h,), 0.1).float()).bfloat16()} for _ in range(case["layers"])]


def attention_inputs(case, seed):
    """q, K and V N(0, 1), the pages of 16 keys in shuffled order."""
    g, pages, kvh = generator(seed), -(-case["ctx"] // PAGE), case["kv_heads"]
    order = torch.randperm(pages, generator=g, device="cuda")
    return order, [(normal(g, (case["q_heads"], HEAD), 1.0), normal(g, (pages, kvh, PAGE, HEAD), 1.0),
                    normal(g, (pages, kvh, HEAD, PAGE), 1.0)) for _ in range(case["layers"])]


def stack_tensors(case, seed):
    """A two-layer checkpoint: projections and embeddings N(0, 0.02), norm weights around 1."""
    m, g = MODELS[case["model"]], generator(seed)
    h, i, q, kv = m["hidden"], m["inter"], m["q_heads"] * HEAD, m["kv_heads"] * HEAD

    def norm(n):
        return (1.0 + normal(g, (n,), 0.1).float()).bfloat16()

    t = {"model.embed_tokens.weight": normal(g, (STACK_VOCAB, h), 0.02)}
    for layer in range(2):
        p = f"model.layers.{layer}."
        t[p + "input_layernorm.weight"] = norm(h)
        t[p + "self_attn.q_proj.weight"] = normal(g, (q, h), 0.02)
        t[p + "self_attn.k_proj.weight"] = normal(g, (kv, h), 0.02)
        t[p + "self_attn.v_proj.weight"] = normal(g, (kv, h), 0.02)
        t[p + "self_attn.q_norm.weight"] = norm(HEAD)
        t[p + "self_attn.k_norm.weight"] = norm(HEAD)
        t[p + "self_attn.o_proj.weight"] = normal(g, (h, q), 0.02)
        t[p + "post_attention_layernorm.weight"] = norm(h)
        t[p + "mlp.gate_proj.weight"] = normal(g, (i, h), 0.02)
        t[p + "mlp.up_proj.weight"] = normal(g, (i, h), 0.02)
        t[p + "mlp.down_proj.weight"] = normal(g, (h, i), 0.02)
    t["model.norm.weight"] = norm(h)
    t["lm_head.weight"] = normal(g, (STACK_VOCAB, h), 0.02)
    return t


def safetensors(tensors):
    header, at, parts = {}, 0, []
    for name, t in tensors.items():
        size = t.numel() * 2
        header[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + size]}
        at += size
        parts.append(memoryview(t.view(torch.int16).cpu().numpy().reshape(-1).view(np.uint8)))
    head = json.dumps(header).encode()
    return b"".join([len(head).to_bytes(8, "little"), head] + parts)


def prompt_ids(seed, shape, vocab):
    return np.random.default_rng(seed).integers(0, vocab, shape, dtype=np.uint32)


def prepare(case, seed):
    if case["kind"] in ("stack", "chat", "batch"):
        return prepare_engine(case, seed)
    return {"linear": prepare_linear, "mlp": prepare_mlp, "attention": prepare_attention}[case["kind"]](case, seed)


def launches(state, calls):
    """A program that decodes records a step's launches once; a single call is made as it is."""
    torch.cuda.synchronize()
    if state["case"]["layers"] > 1:
        state["graph"] = gpu().capture(lambda: [c() for c in calls])
    state["calls"] = calls
    return state


def prepare_linear(case, seed):
    g, rows, cols, n = gpu(), case["rows"], case["cols"], case["n"]
    layers = linear_inputs(case, seed)
    out = [torch.empty((n, rows), dtype=torch.float32 if case["f32"] else torch.bfloat16, device="cuda") for _ in layers]
    calls = [functools.partial(g.gemv, w.data_ptr(), rows, cols, x.data_ptr(), n, y.data_ptr(), case["f32"])
             for (w, x), y in zip(layers, out)]
    return launches({"case": case, "keep": layers, "out": out}, calls)


def prepare_mlp(case, seed):
    g = gpu()
    layers = mlp_inputs(case, seed)
    out = [{"y": torch.empty(case["inter"], dtype=torch.bfloat16, device="cuda"),
            "res_out": torch.empty(case["hidden"], dtype=torch.float32, device="cuda")} for _ in layers]
    calls = [functools.partial(g.gemv_fused, rows=2 * case["inter"], cols=case["hidden"], prologue=NORM, epilogue=SWIGLU,
                               eps=EPS, f64_sums=int(case["exact_sums"]),
                               **{k: v.data_ptr() for k, v in {**i, **o}.items()}) for i, o in zip(layers, out)]
    return launches({"case": case, "keep": layers, "out": out}, calls)


def prepare_attention(case, seed):
    g, qh, kvh, ctx = gpu(), case["q_heads"], case["kv_heads"], case["ctx"]
    order, layers = attention_inputs(case, seed)
    plan = g.split_plan(qh, kvh)
    keep = {"layers": layers, "table": order.to(torch.int32), "pos": torch.tensor([ctx - 1], dtype=torch.int32, device="cuda"),
            "state": torch.empty(split_state_bytes(qh, plan.splits), dtype=torch.uint8, device="cuda"),
            "counter": torch.zeros(kvh, dtype=torch.int32, device="cuda")}
    out = [torch.empty((qh, HEAD), dtype=torch.bfloat16, device="cuda") for _ in layers]
    scale = float(np.float32(1.0 / math.sqrt(HEAD)))
    calls = [functools.partial(g.attention_split, plan, plan.grouped, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                               keep["table"].data_ptr(), keep["state"].data_ptr(), keep["counter"].data_ptr(),
                               o.data_ptr(), keep["pos"].data_ptr(), qh, kvh, ctx, scale)
             for (q, k, v), o in zip(layers, out)]
    return launches({"case": case, "keep": keep, "out": out}, calls)


def prepare_engine(case, seed):
    m = MODELS[case["model"]]
    if case["kind"] == "stack":
        opts = EngineOptions(max_ctx=case["prompt"] + 16, page_seed=seed + 1, f64_sums=None if case["exact_sums"] else False)
        engine = Engine.load_from(config(case["model"], 2, STACK_VOCAB, False),
                                  {"model.safetensors": safetensors(stack_tensors(case, seed))}, opts)
        ids = prompt_ids(seed, case["prompt"], STACK_VOCAB)
    elif case["kind"] == "chat":
        engine = Engine.load_synthetic(config(case["model"], m["layers"], VOCAB, m["tied"]), seed, 0.02,
                                       EngineOptions(max_ctx=case["prompt"] + case["tokens"] + 16, page_seed=seed + 1))
        ids = prompt_ids(seed, case["prompt"], VOCAB)
    else:
        # Tied embeddings and a small scale: each token's own embedding stays visible in the
        # residual, so the greedy tokens have the clear margins of a trained model's.
        engine = Engine.load_synthetic(config(case["model"], m["layers"], VOCAB, True), seed, m["batch_std"],
                                       EngineOptions(max_ctx=case["prompt"] + case["tokens"] + 16, page_seed=seed + 1,
                                                     max_batch=case["batch"]))
        ids = prompt_ids(seed, (case["batch"], case["prompt"]), VOCAB)
    return {"case": case, "engine": engine, "ids": ids}


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        tokens, _, logits = state["engine"].greedy_batch(state["ids"], case["tokens"], logits=True)
        return {"tokens": tokens, "logits": logits}
    if case["kind"] in ("chat", "stack"):
        tokens, logits = state["engine"].greedy_with_last_logits(state["ids"], case.get("tokens", 1))
        return {"tokens": tokens, "logits": logits} if case["kind"] == "chat" else {"logits": logits}
    if "graph" in state:
        gpu().launch_graph(state["graph"])
    else:
        state["calls"][0]()
    return {"out": state["out"]}


# -- what a pass cannot do without --

def layer_params(model):
    return sum(r * c for r, c in projections(model).values())


def work(case):
    kind = case["kind"]
    if kind == "linear":
        rows, cols, n, layers = case["rows"], case["cols"], case["n"], case["layers"]
        return {"bytes": layers * (2 * rows * cols + 2 * n * cols + (4 if case["f32"] else 2) * n * rows),
                "flops": layers * 2 * rows * cols * n}
    if kind == "mlp":
        h, i, layers = case["hidden"], case["inter"], case["layers"]
        return {"bytes": layers * (4 * h * i + 12 * h + 2 * i), "flops": layers * 4 * h * i}
    if kind == "attention":
        qh, kvh, ctx, layers = case["q_heads"], case["kv_heads"], case["ctx"], case["layers"]
        return {"bytes": layers * (2 * ctx * kvh * HEAD * 2 + 4 * qh * HEAD), "flops": layers * 4 * qh * HEAD * ctx}
    m = MODELS[case["model"]]
    depth, vocab = (2, STACK_VOCAB) if kind == "stack" else (m["layers"], VOCAB)
    seqs, prompt, steps = case.get("batch", 1), case["prompt"], case.get("tokens", 1) - 1
    weights = depth * layer_params(case["model"]) + vocab * m["hidden"]
    kv = depth * 2 * m["kv_heads"] * HEAD * 2  # K/V bytes of a position
    pairs = prompt * (prompt + 1) / 2 + sum(prompt + 1 + s for s in range(steps))
    return {"bytes": 2 * weights * (1 + steps) + seqs * kv * (prompt + sum(prompt + 1 + s for s in range(steps))),
            "flops": seqs * (2 * depth * layer_params(case["model"]) * (prompt + steps)
                             + 2 * vocab * m["hidden"] * (1 + steps) + depth * 4 * m["q_heads"] * HEAD * pairs)}


def tolerance(case):
    """About four times what the path's own forms differ by: the few-row and the tiled GEMM, f32
    and f64 sums, other split-K factors, prompts in passes of other lengths, decode steps in the
    place of a pass. The exact sums are the same bits in all of them; one rounding that falls to
    the other side travels through a stack's later layers and through every layer of a model."""
    kind = case["kind"]
    if kind == "linear" and case["f32"]:
        return {"rel": 4e-6, "max": 4e-5}
    if kind in ("linear", "attention"):
        return {"rel": 3e-4, "max": 0.01}  # few of the bf16 results round the other way
    if kind == "mlp":
        return {"rel": 3e-4, "max": 0.02}  # gate and up are rounded before their product
    if kind == "batch":
        return {"rel": 0.016, "max": 0.1, "differ": 0.01}
    if kind == "chat":
        return {"rel": 0.01, "max": 0.1, "differ": 0.01}
    return {"rel": 1e-3, "max": 0.02} if case["exact_sums"] else {"rel": 0.03, "max": 0.15}


# -- the same in 64 bits --

def rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def silu(x):
    return x / (1.0 + torch.exp(-x))


def exact_linear(case, seed):
    return {"out": [x.double() @ w.double().T for w, x in linear_inputs(case, seed)]}


def exact_mlp(case, seed):
    out = []
    for i in mlp_inputs(case, seed):
        res = i["res_in"].double() + i["delta"].double()
        gu = i["w"].double() @ rms(res, i["norm_w"])
        out.append({"y": silu(gu[:case["inter"]]) * gu[case["inter"]:], "res_out": res})
    return {"out": out}


def exact_attention(case, seed):
    order, layers = attention_inputs(case, seed)
    qh, kvh, ctx, out = case["q_heads"], case["kv_heads"], case["ctx"], []
    for q, k, v in layers:
        keys = k[order].double().permute(1, 0, 2, 3).reshape(kvh, -1, HEAD)[:, :ctx]
        vals = v[order].double().permute(1, 0, 3, 2).reshape(kvh, -1, HEAD)[:, :ctx]
        s = q.double().view(kvh, qh // kvh, HEAD) @ keys.transpose(1, 2).contiguous() / math.sqrt(HEAD)
        out.append((torch.softmax(s, -1) @ vals).reshape(qh, HEAD))
    return {"out": out}


def exact_stack(case, seed):
    m, t = MODELS[case["model"]], stack_tensors(case, seed)
    qh, kvh, n = m["q_heads"], m["kv_heads"], case["prompt"]
    group = qh // kvh
    ids = torch.from_numpy(prompt_ids(seed, n, STACK_VOCAB).astype(np.int64)).cuda()
    inv = 1.0 / THETA ** (torch.arange(0, HEAD, 2, dtype=torch.float64, device="cuda") / HEAD)
    angle = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * inv
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rope(x):
        a, b = x[..., :HEAD // 2], x[..., HEAD // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    r = t["model.embed_tokens.weight"][ids].double()
    for layer in range(2):
        def w(name, p=f"model.layers.{layer}."):
            return t[p + name + ".weight"]

        def proj(x, name):
            return x @ w(name).double().T.contiguous()

        x = rms(r, w("input_layernorm"))
        q = rope(rms(proj(x, "self_attn.q_proj").view(n, qh, HEAD), w("self_attn.q_norm")))
        k = rope(rms(proj(x, "self_attn.k_proj").view(n, kvh, HEAD), w("self_attn.k_norm")))
        v = proj(x, "self_attn.v_proj").view(n, kvh, HEAD)
        o = torch.empty((n, qh, HEAD), dtype=torch.float64, device="cuda")
        for row in range(0, n, 1024):
            end = min(n, row + 1024)
            hidden = torch.arange(end, device="cuda")[None] > torch.arange(row, end, device="cuda")[:, None]
            for head in range(qh):
                s = q[row:end, head] @ k[:end, head // group].T.contiguous() / math.sqrt(HEAD)
                o[row:end, head] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:end, head // group]
        r = r + proj(o.reshape(n, -1), "self_attn.o_proj")
        if layer == 1:
            r = r[-1:]
        x = rms(r, w("post_attention_layernorm"))
        r = r + proj(silu(proj(x, "mlp.gate_proj")) * proj(x, "mlp.up_proj"), "mlp.down_proj")
    return {"logits": (rms(r, t["model.norm.weight"]) @ t["lm_head.weight"].double().T.contiguous())[0]}


def exact(case, seed):
    """run()'s outputs in 64 bits without any rounding in between; None for a whole model."""
    if case["kind"] in ("chat", "batch"):
        return None
    return {"linear": exact_linear, "mlp": exact_mlp, "attention": exact_attention, "stack": exact_stack}[case["kind"]](case, seed)
