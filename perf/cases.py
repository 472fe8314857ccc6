"""The work that users of this framework have it do, as cases that can be timed and checked.

A case is one request pattern of the generation API on one model: ``prepare`` loads random weights into an engine and fills the
caches, ``run`` is the request, ``exact`` is the same request in 64-bit torch.  Models are the shapes that this repository's
benchmark uses (or generic ones), at a depth that keeps preparation quick; every layer costs the same, so depth only scales a
pass.  Weights are N(0, 1.6 / width) -- 0.02^2 at 4096 -- with the usual 1 / sqrt(2 layers) on the matrices that write to the
residual stream.  Where a case feeds sampled tokens back, the output matrix favours one successor of every token, as a trained
model's does: without that two correct implementations in 16 bits part at the first near-tie and what follows cannot be
compared.  Where it cannot (a tied output matrix, nucleus sampling), given tokens are fed instead.
"""
from __future__ import annotations

import math

import numpy as np
import torch

MISTRAL_7B = dict(arch="llama", hidden=4096, heads=32, kv_heads=8, head_dim=128, ff=14336, vocab=32000, eps=1e-5, theta=10000.0, tied=False)
QWEN3_14B = dict(arch="qwen3", hidden=5120, heads=40, kv_heads=8, head_dim=128, ff=17408, vocab=151936, eps=1e-6, theta=1000000.0, tied=False)
TINY = dict(arch="llama", hidden=64, heads=4, kv_heads=4, head_dim=16, ff=128, vocab=151936, eps=1e-6, theta=10000.0, tied=True)
RUNEVIK = dict(arch="runevik", hidden=2048, heads=16, kv_heads=8, head_dim=128, ff=8192, vocab=32000, eps=1e-5, tied=False, kv_rank=512, conv=4, side=64)
BLOCK_TOKENS = 64                      # of the block-paged caches: the server's
TOP_LOGPROBS = 5                       # where a case asks for logprobs
LORA_RANK, LORA_SCALE = 16, 10.0


def case(name, model, layers, kind, batch, context, steps, bits=0, dtype="bfloat16", kv="model", top_p=0.0, lora=0, chunk=0):
    """kind: "decode" (`steps` tokens for each of `batch` sequences whose prompts are in the cache), "generate" (prompt and `steps`
    tokens), "prefill" (prompts only), "score" (log-probabilities of given tokens), "mixed" (`steps` steps that decode
    `batch` sequences and take in `chunk` tokens of a new prompt each).  bits = 0: dense weights."""
    return dict(model, **({"name": name} if name else {}), layers=layers, kind=kind, batch=batch, context=context, steps=steps, bits=bits, dtype=dtype,
                kv=kv, top_p=top_p, lora=lora, chunk=chunk)


def listed():
    return [
        # a smoke-test model, two short prompts: nothing but launches and host work
        case("tiny_generate_b2", TINY, 8, "generate", 2, 9, 16, bits=4, kv="float32"),
        # one user chatting with a 16-bit model: the latency of a token
        case("chat_b1", MISTRAL_7B, 8, "decode", 1, 321, 16),
        # the headline benchmark: eight sequences at 1024 tokens, the reference's float32 caches, the whole model
        case("decode_b8_kv32", MISTRAL_7B, 32, "decode", 8, 1025, 8, kv="float32"),
        # a 4-bit model on the same load, nucleus sampling with log-probabilities
        case("decode_b8_int4_topp", MISTRAL_7B, 16, "decode", 8, 1025, 8, bits=4, top_p=0.9),
        # a few requests of odd length from prompt to answer, 8-bit weights, contiguous caches
        case("generate_b3_int8", MISTRAL_7B, 8, "generate", 3, 333, 16, bits=8),
        # a server's batch on a larger 16-bit model
        case("decode_b32", QWEN3_14B, 8, "decode", 32, 1025, 8),
        # the largest server batch: 4-bit weights with an adapter
        case("decode_b64_int4_lora", QWEN3_14B, 10, "decode", 64, 513, 8, bits=4, lora=2),
        # continuous batching: live sequences decode while a prompt comes in piece by piece
        case("mixed_b31_int4", QWEN3_14B, 8, "mixed", 31, 641, 4, bits=4, chunk=32),
        # prompts of a full batch, float32 caches
        case("prefill_8x1024_kv32", MISTRAL_7B, 8, "prefill", 8, 1024, 0, kv="float32"),
        # perplexity of one document on a 4-bit model: every position's logits
        case("score_700_int4", MISTRAL_7B, 8, "score", 1, 700, 0, bits=4),
        # long documents in the cache, half-precision weights: the attention counts
        case("decode_b4_long_f16", MISTRAL_7B, 8, "decode", 4, 8001, 8, dtype="float16"),
        # a layer-list model (recurrent and latent layers) from prompt to answer
        case("runevik_generate_b4", RUNEVIK, 8, "generate", 4, 500, 16),
    ]


def draw(rng):
    """A case of the same kinds, sizes between the smallest and the largest listed ones."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if rng.random() < 0.12:
        return case(None, dict(RUNEVIK, hidden=rng.choice([1024, 2048])), 4, "generate", spread(1, 8), spread(16, 700), spread(4, 16))
    heads, group = rng.choice([(8, 1), (16, 4), (16, 8), (24, 4), (32, 4), (40, 5)])
    generic = dict(arch=rng.choice(["llama", "qwen3"]), hidden=heads * 128, heads=heads, kv_heads=heads // group, head_dim=128,
                   ff=64 * int(heads * 128 * rng.uniform(2.6, 4.0) / 64), vocab=rng.choice([32000, 50304, 128256]), eps=1e-5, theta=10000.0, tied=False)
    model = rng.choice([MISTRAL_7B, QWEN3_14B, generic, generic])
    kind = rng.choice(["decode", "decode", "decode", "generate", "prefill", "score", "mixed"])
    bits, dtype, kv = rng.choice([0, 0, 4, 4, 8]), rng.choice(["bfloat16", "bfloat16", "float16"]), rng.choice(["model", "model", "float32"])
    layers, steps = rng.randint(3, 8), spread(4, 16)
    if kind == "decode":
        batch = spread(1, 64)
        context = 64 * max(1, spread(40, max(64, min(8000, 32000 // batch))) // 64) + rng.choice([1, 1, 6])
        return case(None, model, layers, kind, batch, context, steps, bits, dtype, kv, top_p=rng.choice([0.0, 0.0, 0.9]), lora=1 if rng.random() < 0.2 else 0)
    if kind == "generate":
        batch = spread(1, 16)
        return case(None, model, layers, kind, batch, spread(8, min(1000, 4000 // batch)), steps, bits, dtype, kv)
    if kind == "mixed":
        batch = spread(2, 40)
        return case(None, model, layers, kind, batch, 64 * max(1, spread(64, 16000 // batch) // 64) + 1, 4, bits, dtype, kv, chunk=rng.choice([16, 32, 64, 200]))
    batch = spread(1, 8)
    return case(None, model, layers, kind, batch, spread(32, min(2000, (6000 if kind == "prefill" else 1500) // batch)), 0, bits, dtype, kv)


# ---- models ------------------------------------------------------------------------------------------------------------------

def config(c):
    if c["arch"] == "runevik":
        W, H = c["hidden"], c["hidden"] // 128
        delta = {"type": "delta", "mlp": {"ff": 4 * W, "kind": "dense"}, "mixer": {"heads": H, "kv_heads": H // 2, "dim": 128, "vdim": 128, "conv": c["conv"]}}
        lat = {"type": "latent_attention", "mlp": {"ff": 4 * W, "kind": "dense"},
               "mixer": {"heads": H, "dim": 128, "vdim": 128, "kv_rank": min(c["kv_rank"], W // 4), "scale": 128 ** -0.5}}
        return {"model_type": "runevik", "architecture": "Runevik", "width": W, "vocab": c["vocab"], "norm": {"eps": c["eps"]},
                "layers": [lat if i % 4 == 3 else delta for i in range(c["layers"])], "token_side": {"dim": c["side"]}}
    cfg = dict(model_type=c["arch"], hidden_size=c["hidden"], num_hidden_layers=c["layers"], num_attention_heads=c["heads"],
               num_key_value_heads=c["kv_heads"], head_dim=c["head_dim"], intermediate_size=c["ff"], vocab_size=c["vocab"], rms_norm_eps=c["eps"],
               rope_theta=c["theta"], tie_word_embeddings=c["tied"], max_position_embeddings=16384)
    if c["bits"]:
        cfg["quantization"] = {"bits": c["bits"], "group_size": 64}
    return cfg


def specs(c):
    """(name, shape, standard deviation or None for a weight around one) of every tensor, in a fixed order."""
    W, V, std = c["hidden"], c["vocab"], 1.28 / math.sqrt(c["hidden"])
    back = std / math.sqrt(2 * c["layers"])
    if c["arch"] == "runevik":
        yield "embed", (V, W), 1.0
        yield "side.embed", (V, c["side"] * c["layers"]), 1.0
        for i, layer in enumerate(config(c)["layers"]):
            p, m, H = f"l{i}.", layer["mixer"], W // 128
            yield p + "norm1", (), None
            if layer["type"] == "delta":
                for t, n in (("q", H * 64), ("k", H * 64), ("v", W)):
                    yield p + "mix." + t, (n, W), std
                    yield p + f"mix.{t}.conv", (n, m["conv"]), 0.5
                yield p + "mix.g", (W, W), std
                yield p + "mix.a", (H, W), std
                yield p + "mix.b", (H, W), std
                yield p + "mix.A_log", (H,), 0.5
                yield p + "mix.dt_bias", (H,), 1.0
                yield p + "mix.norm", (128,), None
            else:
                yield p + "mix.q", (W, W), std
                yield p + "mix.dkv", (m["kv_rank"], W), std
                yield p + "mix.dkv.norm", (m["kv_rank"],), None
                yield p + "mix.uk", (W, m["kv_rank"]), std
                yield p + "mix.uv", (W, m["kv_rank"]), std
                yield p + "mix.g", (H, W), std
            yield p + "mix.o", (W, W), back
            yield p + "mlp.up", (4 * W, W), std
            yield p + "mlp.down", (W, 4 * W), back
            yield p + "mlp.act", (4,), None
            yield p + "side.gate", (c["side"], W), std
            yield p + "side.proj", (W, c["side"]), 0.1
            yield p + "side.norm", (W,), 0.1
        yield "final.norm", (), None
        yield "head", (V, W), std
        return
    nq, nkv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    yield "model.embed_tokens.weight", (V, W), std if c["tied"] else 1.0
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        yield p + "self_attn.q_proj.weight", (nq, W), std
        yield p + "self_attn.k_proj.weight", (nkv, W), std
        yield p + "self_attn.v_proj.weight", (nkv, W), std
        yield p + "self_attn.o_proj.weight", (W, nq), back
        if c["arch"] == "qwen3":
            yield p + "self_attn.q_norm.weight", (c["head_dim"],), None
            yield p + "self_attn.k_norm.weight", (c["head_dim"],), None
        yield p + "mlp.gate_proj.weight", (c["ff"], W), std
        yield p + "mlp.up_proj.weight", (c["ff"], W), std
        yield p + "mlp.down_proj.weight", (W, c["ff"]), back
        yield p + "input_layernorm.weight", (W,), None
        yield p + "post_attention_layernorm.weight", (W,), None
    yield "model.norm.weight", (W,), None
    if not c["tied"]:
        yield "lm_head.weight", (V, W), std


def forced(c):
    """Whether given tokens are fed (see above); sampled ids are then no output: they move with the last bit of a logit."""
    return bool(c["top_p"] or c["tied"])


def draw_tensor(c, seed, name, shape, std):
    gen = torch.Generator(device="cuda").manual_seed((seed * 1000003 + sum(ord(ch) * 31 ** k for k, ch in enumerate(name))) % (1 << 62))
    dt = getattr(torch, c["dtype"])
    t = torch.randn(shape, generator=gen, device="cuda", dtype=dt)
    return t.mul_(0.1).add_(1.0) if std is None else t.mul_(std)


def tensors(c, seed):
    """(name, tensor in the model's type) of the whole model, one at a time."""
    embed = None
    for name, shape, std in specs(c):
        t = draw_tensor(c, seed, name, shape, std)
        if name in ("model.embed_tokens.weight", "embed"):
            embed = t
        if name in ("lm_head.weight", "head") and not forced(c):       # the successor of token v: row (v + 1) mod vocab
            t.add_(torch.roll(embed, 1, 0), alpha=(80.0 if c["arch"] == "runevik" else 20.0) / c["hidden"])
        yield name, t


def quantized(c, w):
    """Affine groups of 64 along the inputs: w ~ scale * code + bias, 32 / bits codes per word, little-endian.  -> words, scales, biases"""
    n, k = w.shape
    top, per = (1 << c["bits"]) - 1, 32 // c["bits"]
    g = w.float().view(n, k // 64, 64)
    lo, hi = g.amin(-1), g.amax(-1)
    scale, bias = ((hi - lo) / top).to(w.dtype), lo.to(w.dtype)
    code = ((g - bias.float()[..., None]) / scale.float()[..., None]).round_().clamp_(0, top).to(torch.int32).view(n, k // per, per)
    words = code[..., 0].clone()
    for j in range(1, per):
        words |= code[..., j] << (j * c["bits"])
    return words, scale, bias


def adapters(c, seed):
    """(layer, projection, A, B) of the low-rank adapters on the last layers' queries and values."""
    for layer in range(c["layers"] - c["lora"], c["layers"]):
        for proj, n in (("self_attn.q_proj", c["heads"] * c["head_dim"]), ("self_attn.v_proj", c["kv_heads"] * c["head_dim"])):
            gen = torch.Generator(device="cuda").manual_seed(seed * 7919 + 2 * layer + (n != c["heads"] * c["head_dim"]) + 17)
            a = torch.rand((c["hidden"], LORA_RANK), generator=gen, device="cuda").mul_(2).sub_(1).div_(math.sqrt(c["hidden"]))
            yield layer, proj, a, torch.randn((LORA_RANK, n), generator=gen, device="cuda").mul_(0.01)


def is_matrix(shape):
    return len(shape) == 2


def inputs(c, seed):
    """Token ids: prompts [rows][context] (mixed: one row more, the arriving prompt), the tokens fed afterwards [rows][steps + 1]."""
    rng = np.random.default_rng(seed)
    rows = c["batch"] + (c["kind"] == "mixed")
    prompts = rng.integers(0, c["vocab"], (rows, c["context"])).astype(np.int32)
    return prompts, rng.integers(0, c["vocab"], (rows, max(c["steps"] + 1, 1 + c["steps"] * c["chunk"], c["context"]))).astype(np.int32)


def prepare(c, seed):
    from mlx_parallm_amd.engine import Engine

    limit = c["context"] + c["steps"] * max(1, c["chunk"]) + 2 * BLOCK_TOKENS
    engine = Engine(config(c), device=0, max_positions=limit, act_dtype=c["dtype"])
    for name, t in tensors(c, seed):
        if c["bits"] and is_matrix(t.shape):
            for part, x in zip((".weight", ".scales", ".biases"), quantized(c, t)):
                engine.set_tensor(name[: -len(".weight")] + part, x)
        else:
            engine.set_tensor(name, t)
    engine.finalize()
    for layer, proj, a, b in adapters(c, seed):
        engine.set_lora(layer, proj, a, b, LORA_SCALE)
    prompts, fed = inputs(c, seed)
    state = {"case": c, "engine": engine, "prompts": prompts, "fed": fed}
    rows = len(prompts)
    if c["kind"] in ("decode", "mixed"):
        kv = engine.new_paged_kv(rows, block_tokens=BLOCK_TOKENS, max_tokens_per_row=limit, kv_dtype=c["kv"])
        full = c["context"] // BLOCK_TOKENS * BLOCK_TOKENS      # what a server's prefix cache keeps of the prompts
        group = max(1, 8192 // max(1, full))
        for r in range(0, rows, group) if full else ():
            some = list(range(r, min(rows, r + group)))
            for at in range(0, full, 4096):
                part = prompts[some, at:min(full, at + 4096)]
                engine.step_wait(engine.step_enqueue_rows(kv, some, part), len(some))
        for r in range(rows):
            kv.prefix_publish(r, prompts[r, :full])
        state["kv"] = kv
    else:
        state["kv"] = engine.new_kv(rows, capacity=min(limit, c["context"] + c["steps"] + 2), kv_dtype=c["kv"])
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------------------

def sampling(c, step):
    from mlx_parallm_amd.engine import SampleArgs

    if c["top_p"]:
        return SampleArgs(temp=1.0, top_p=c["top_p"], seed=1234, top_logprobs=TOP_LOGPROBS, stream_position=step)
    return SampleArgs(temp=0.0)


def run(state):
    c, engine, kv, prompts, fed = (state[k] for k in ("case", "engine", "kv", "prompts", "fed"))
    B = c["batch"]
    if c["kind"] == "prefill":
        kv.reset()
        return {"logits": engine.forward(prompts, kv)}
    if c["kind"] == "score":
        from mlx_parallm_amd.engine import SampleArgs

        kv.reset()
        r = engine.score_tokens(kv, prompts, fed[:, :c["context"]], SampleArgs(top_logprobs=TOP_LOGPROBS))
        return {"logprobs": r["logprobs"], "top_logprobs": r["top_logprobs"]}
    if c["kind"] == "mixed":
        return run_mixed(c, engine, kv, prompts, fed)
    if c["kind"] == "generate":
        kv.reset()
        ticket = engine.step_enqueue(kv, prompts, sampling(c, 0))
    else:                                            # the prompts come from the prefix cache, but for what fills no block
        left = 0
        for r in range(B):
            kv.reset_row(r)
            left = kv.prefix_attach(r, prompts[r])
        ticket = engine.step_enqueue(kv, prompts[:, left:], sampling(c, 0))
    out = []
    for step in range(1, c["steps"]):                # the next step is enqueued before the last one's tokens are read
        after = engine.step_enqueue(kv, fed[:B, step:step + 1] if forced(c) else None, sampling(c, step))
        out.append(engine.step_wait(ticket, B, TOP_LOGPROBS if c["top_p"] else 0))
        ticket = after
    out.append(engine.step_wait(ticket, B, TOP_LOGPROBS if c["top_p"] else 0))
    result = {"logprobs": np.stack([r["logprobs"] for r in out], 1)}
    if c["top_p"]:
        result["top_logprobs"] = np.stack([r["top_logprobs"] for r in out], 1)
    if not forced(c):
        result["tokens"] = np.stack([r["tokens"] for r in out], 1)
    result["logits"] = engine.forward(fed[:B, c["steps"]:c["steps"] + 1] if forced(c) else result["tokens"][:, -1:], kv)
    return result


def run_mixed(c, engine, kv, prompts, fed):
    B, chunk = c["batch"], c["chunk"]
    for r in range(B + 1):
        kv.reset_row(r)
        left = kv.prefix_attach(r, prompts[r])
    live, coming, tokens, logprobs = list(range(B)), fed[B], [], []
    tail = [prompts[r, left:] for r in range(B + 1)]
    if len(tail[0]) > 1:
        engine.forward_segments(kv, live, [t[:-1] for t in tail[:B]])
    now = [t[-1:] for t in tail[:B]]
    pieces = [np.concatenate([tail[B], coming])[i * chunk:(i + 1) * chunk] for i in range(c["steps"])]
    for i, piece in enumerate(pieces[:-1]):
        r = engine.step_wait(engine.step_enqueue_mixed(kv, live + [B], now + [piece], [1] * B + [0], sampling(c, i)), B)
        tokens.append(r["tokens"])
        logprobs.append(r["logprobs"])
        now = [t[None] for t in (fed[:B, i + 1] if forced(c) else r["tokens"])]
    logits = engine.forward_segments(kv, live + [B], now + [pieces[-1]], list(range(B)) + [B + len(pieces[-1]) - 1])
    return {"logprobs": np.stack(logprobs, 1), "logits": logits, **({} if forced(c) else {"tokens": np.stack(tokens, 1)})}


# ---- what a pass cannot do without -------------------------------------------------------------------------------------------

def work(c):
    bits = {0: 16.0, 4: 4.5, 8: 8.5}[c["bits"]]                 # with a scale and a bias per 64 weights
    size = {name: math.prod(shape) for name, shape, _ in specs(c) if is_matrix(shape) and not name.endswith("side.embed")}
    head = size.pop("head" if c["arch"] == "runevik" else "lm_head.weight" if not c["tied"] else "model.embed_tokens.weight")
    size.pop("embed", None), size.pop("model.embed_tokens.weight", None)
    body = sum(size.values())
    kvb = 4 if c["kv"] == "float32" else 2
    if c["arch"] == "runevik":       # latents of every fourth layer; the states of the others are read and written
        attn = c["layers"] // 4
        kv_tok, state, qk = attn * min(c["kv_rank"], c["hidden"] // 4) * kvb, (c["layers"] - attn) * c["hidden"] * 128 * 4 * 2, attn * c["hidden"]
    else:
        kv_tok, state, qk = 2 * c["layers"] * c["kv_heads"] * c["head_dim"] * kvb, 0, c["layers"] * c["heads"] * c["head_dim"]
    total = {"bytes": 0.0, "flops": 0.0}

    def one(rows, new, before, heads):                          # a pass over the weights: `new` tokens on `before` cached ones, for each row
        total["bytes"] += (body + head * (heads > 0)) * bits / 8 + rows * (before + new) * kv_tok + rows * new * 4 + heads * c["vocab"] * 4 + rows * state
        total["flops"] += 2.0 * rows * new * body + 2.0 * heads * head + 4.0 * rows * new * (before + (new + 1) / 2) * qk

    B, L = c["batch"], c["context"]
    kept = 0 if c["kind"] == "generate" else (L - 1) // BLOCK_TOKENS * BLOCK_TOKENS        # tokens of a prompt that are in the cache
    if c["kind"] == "prefill":
        one(B, L, 0, B)
    elif c["kind"] == "score":
        one(B, L, 0, B * L)
    elif c["kind"] == "mixed":
        if L - kept > 1:
            one(B, L - kept - 1, kept, 0)
        for i in range(c["steps"]):
            one(B, 1, L - 1 + i, B)
            total["flops"] += 2.0 * c["chunk"] * body
            total["bytes"] += (kept + (i + 1) * c["chunk"]) * kv_tok
    else:
        one(B, L - kept, kept, B)
        for i in range(c["steps"]):
            one(B, 1, L + i, B)
    return total


def tolerance(c):
    """About four times what the path is off from 64 bits (logits 1.0 to 1.6e-2 in bfloat16, 1.1 to 3.0e-3 in float16), and no more than
    3e-2.  With float32 caches the first layer still rounds to 16 bits, the rest does not: 4e-4 to 3.6e-3 off, the smoke-test model
(sums of 64 terms, weights of 4 bits) 1.3 to 2.2e-2."""
    if c["kv"] == "float32" and c["hidden"] >= 1024:
        return {"rel": 0.01, "max": 0.1, "differ": 0.01}
    return {"rel": 0.012, "max": 0.12, "differ": 0.01} if c["dtype"] == "float16" else {"rel": 0.03, "max": 0.3, "differ": 0.01}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------

def exact_weights(c, seed):
    """The model's tensors in float64 by name: as the engine got them (codes, scales and biases multiplied out)."""
    kept = {}
    for name, t in tensors(c, seed):
        if c["bits"] and is_matrix(t.shape):
            words, scale, bias = quantized(c, t)
            code = torch.stack([(words >> (j * c["bits"])) & ((1 << c["bits"]) - 1) for j in range(32 // c["bits"])], -1)
            t = (code.view(t.shape[0], -1, 64) * scale[..., None].float() + bias[..., None].float()).view(t.shape)      # (exact: few significant bits)
        kept[name] = t
    return kept


def rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def rotate(x, at, theta):
    """x [rows][heads][tokens][dim], at [tokens]: coordinate i and i + dim / 2 turn by position * theta^(-2 i / dim)."""
    half = x.shape[-1] // 2
    angle = at.double()[:, None] * theta ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], -1)


def attend(q, k, v, before, scale):
    """q [rows][heads][tokens][dim] behind `before` cached tokens, k, v [rows][kv heads][before + tokens][dim]."""
    out, group = torch.empty_like(q), q.shape[1] // k.shape[1]
    block = max(1, int(4e8 // (k.shape[2] * group)))
    keys = torch.arange(k.shape[2], device=q.device)
    for r in range(q.shape[0]):
        for g in range(k.shape[1]):
            for t in range(0, q.shape[2], block):
                qq = q[r, g * group:(g + 1) * group, t:t + block]
                s = torch.matmul(qq, k[r, g].T) * scale
                s.masked_fill_(keys[None, None] > torch.arange(t, t + qq.shape[1], device=q.device)[None, :, None] + before, -math.inf)
                out[r, g * group:(g + 1) * group, t:t + block] = torch.matmul(s.softmax(-1), v[r, g])
    return out


def exact_llama(c, w, lora, tokens, cache, before):
    """tokens [rows][n] behind `before` cached ones -> final hidden states [rows][n][hidden] (normed)."""
    R, n = tokens.shape
    H, G, D = c["heads"], c["kv_heads"], c["head_dim"]
    at = torch.arange(before, before + n, device="cuda")
    x = w["model.embed_tokens.weight"][tokens].double()
    for i in range(c["layers"]):
        p = f"model.layers.{i}."

        def lin(y, name):
            z = y @ w[p + name + ".weight"].double().T
            if (i, name) in lora:
                a, b = lora[(i, name)]
                z = z + LORA_SCALE * (y @ a.double() @ b.double())
            return z

        h = rms(x, c["eps"]) * w[p + "input_layernorm.weight"].double()
        q, k, v = (lin(h, f"self_attn.{t}_proj").view(R, n, -1, D).transpose(1, 2) for t in "qkv")
        if c["arch"] == "qwen3":
            q, k = (rms(y, c["eps"]) * w[p + f"self_attn.{t}_norm.weight"].double() for y, t in ((q, "q"), (k, "k")))
        q, k = rotate(q, at, c["theta"]), rotate(k, at, c["theta"])
        if i in cache:
            k, v = torch.cat([cache[i][0], k], 2), torch.cat([cache[i][1], v], 2)
        cache[i] = (k, v)
        x = x + lin(attend(q, k, v, before, D ** -0.5).transpose(1, 2).reshape(R, n, H * D), "self_attn.o_proj")
        h = rms(x, c["eps"]) * w[p + "post_attention_layernorm.weight"].double()
        x = x + lin(torch.nn.functional.silu(lin(h, "mlp.gate_proj")) * lin(h, "mlp.up_proj"), "mlp.down_proj")
    return rms(x, c["eps"]) * w["model.norm.weight"].double()


def exact_runevik(c, w, lora, tokens, cache, before):
    R, n = tokens.shape
    W, H, eps = c["hidden"], c["hidden"] // 128, c["eps"]
    at = torch.arange(before, before + n, device="cuda").double()
    angle = at[:, None] * 10000.0 ** (-torch.arange(0, W, 2, device="cuda").double() / W)
    x = w["embed"][tokens].double() + torch.stack([angle.sin(), angle.cos()], -1).view(n, W)

    def lin(y, name):
        return y @ w[name].double().T

    for i, layer in enumerate(config(c)["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        h = rms(x, eps) * w[f"l{i}.norm1"].double()
        if layer["type"] == "delta":
            S, tail = cache.get(i, (torch.zeros(R, H, 128, 128, device="cuda", dtype=torch.float64), {}))
            past, parts = {}, {}
            for t in "qkv":
                z = lin(h, p + t)
                z = torch.cat([tail[t] if t in tail else z.new_zeros(R, c["conv"] - 1, z.shape[-1]), z], 1)
                past[t] = z[:, z.shape[1] - (c["conv"] - 1):]
                taps = w[p + t + ".conv"].double()
                parts[t] = torch.nn.functional.silu(sum(z[:, j:j + n] * taps[:, j] for j in range(c["conv"]))).view(R, n, -1, 128)
            q, k, v = parts["q"], parts["k"], parts["v"]
            q, k = ((y * torch.rsqrt(y.square().sum(-1, keepdim=True) + 1e-6)).repeat_interleave(2, 2) for y in (q, k))
            q = q * 128 ** -0.5
            beta = lin(h, p + "b").sigmoid()
            decay = (-w[p + "A_log"].double().exp() * torch.nn.functional.softplus(lin(h, p + "a") + w[p + "dt_bias"].double())).exp()
            o = torch.empty_like(v)
            for t in range(n):
                S = S * decay[:, t, :, None, None]
                u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
                S = S + k[:, t, :, :, None] * u[:, :, None, :]
                o[:, t] = (S * q[:, t, :, :, None]).sum(2)
            cache[i] = (S, past)
            o = rms(o, eps) * w[p + "norm"].double() * torch.nn.functional.silu(lin(h, p + "g")).view(R, n, H, 128)
        else:
            lat = rms(lin(h, p + "dkv"), eps) * w[p + "dkv.norm"].double()
            lat = torch.cat([cache[i], lat], 1) if i in cache else lat
            cache[i] = lat
            k, v = (lin(lat, p + t).view(R, -1, H, 128).transpose(1, 2) for t in ("uk", "uv"))
            o = attend(lin(h, p + "q").view(R, n, H, 128).transpose(1, 2), k, v, before, m["scale"]).transpose(1, 2) * lin(h, p + "g").sigmoid()[..., None]
        z = lin(h, f"l{i}.mlp.up")
        a = w[f"l{i}.mlp.act"].double()
        z = a[0] * rms(z, eps) + a[1] * rms(z.square(), eps) + a[2] * rms(z ** 3, eps) + a[3]
        x = x + lin(o.reshape(R, n, W), p + "o") + lin(z, f"l{i}.mlp.down")
        e = w["side.embed"][tokens].double()[..., i * c["side"]:(i + 1) * c["side"]]
        y = lin(torch.nn.functional.gelu(lin(x, f"l{i}.side.gate"), approximate="tanh") * e, f"l{i}.side.proj")
        x = x + rms(y, eps) * w[f"l{i}.side.norm"].double()
    return rms(x, eps) * w["final.norm"].double()


def exact(c, seed):
    w = exact_weights(c, seed)
    lora = {(layer, proj): (a, b) for layer, proj, a, b in adapters(c, seed)}
    stack = exact_runevik if c["arch"] == "runevik" else exact_llama
    head = w["head"] if c["arch"] == "runevik" else w["model.embed_tokens.weight"] if c["tied"] else w["lm_head.weight"]
    prompts, fed = (torch.from_numpy(x).long().cuda() for x in inputs(c, seed))

    def logits(h):
        return torch.cat([h.reshape(-1, h.shape[-1]) @ head[v:v + 16384].double().T for v in range(0, head.shape[0], 16384)], -1).view(*h.shape[:-1], -1)

    def rows(some):
        """The sequences `some`, which nothing couples: what run() returns of them, as a list of [rows][..] arrays."""
        cache, before = {}, 0

        def feed(tokens):
            nonlocal before
            for at in range(0, tokens.shape[1], 2048):
                h = stack(c, w, lora, tokens[:, at:at + 2048], cache, before)
                before += h.shape[1]
            return h

        tok = prompts[some]
        if c["kind"] == "prefill":
            return {"logits": logits(feed(tok)[:, -1])}
        if c["kind"] == "score":
            lp = logits(feed(tok)).log_softmax(-1)
            return {"logprobs": lp.gather(-1, fed[some, :c["context"], None])[..., 0], "top_logprobs": lp.topk(TOP_LOGPROBS, -1)[0]}
        out = {"logprobs": [], **({"top_logprobs": []} if c["top_p"] else {}), **({} if forced(c) else {"tokens": []})}
        arriving = c["kind"] == "mixed" and some[0] == c["batch"]
        if arriving:
            kept = (c["context"] - 1) // BLOCK_TOKENS * BLOCK_TOKENS
            tok = torch.cat([tok, fed[some]], 1)[:, :kept + c["steps"] * c["chunk"]]
            return {"logits": logits(feed(tok)[:, -1])}
        z = logits(feed(tok)[:, -1])
        for step in range(1, c["steps"] + (c["kind"] != "mixed")):
            lp = z.log_softmax(-1)
            best, ids = lp.max(-1)
            out["logprobs"].append(best)
            if c["top_p"]:
                out["top_logprobs"].append(lp.topk(TOP_LOGPROBS, -1)[0])
            if not forced(c):
                out["tokens"].append(ids.int())
            z = logits(feed(fed[some, step:step + 1] if forced(c) else ids[:, None])[:, -1])
        return {"logits": z, **{k: torch.stack(v, 1) for k, v in out.items()}}

    per = max(1, 8300 // c["context"])
    parts = [rows(list(range(r, min(c["batch"], r + per)))) for r in range(0, c["batch"], per)]
    result = {k: torch.cat([p[k] for p in parts]) for k in parts[0]}
    if c["kind"] == "mixed":
        result["logits"] = torch.cat([result["logits"], rows([c["batch"]])["logits"]])
    if c["top_p"]:
        result["logprobs"] = None                    # (of sampled ids)
    return result
