"""The work that this engine's speed is judged by: requests through the step function, prompts first and then token by token.

A pass announces nothing and keeps nothing: the prompts of a case enter in one step, every request then takes its next tokens one a
step beside the others, and all of them end.  It returns the logits that a program which generates or
scores text reads: one row a request at the end of its prompt and one after every decoded token.  The models are the engine's
seven designs at the sizes that ``bench.py`` measures them at, their weights drawn on the GPU from the seed.

``exact`` computes the same logits in 64 bits with torch alone: the weights from their published recurrence, every mechanism as its
formula, token by token where a design is recurrent.
"""
from __future__ import annotations

import hashlib
import json
import math
import tempfile
from pathlib import Path

import numpy as np
import torch

PAGE = 64
STEP_TOKENS = 4096                 # the engine's own budget of a step, which no case's prompts exceed
# (width, q heads, kv heads, feed-forward) of the designs; heads of 128, eight layers, vocabulary 32,768.
SIZES = {"1k": (1024, 8, 2, 3072), "2k": (2048, 16, 4, 6144), "4k": (4096, 32, 8, 12288)}
LAYERS, VOCAB = 8, 32768
# (width, layers, q heads, feed-forward, tied head) of the Qwen3 shapes; 8 kv heads of 128, vocabulary 151,936, all layers.
QWEN3 = {"0.6b": (1024, 28, 16, 3072, True), "1.7b": (2048, 28, 16, 6144, True), "4b": (2560, 36, 32, 9728, True),
         "8b": (4096, 36, 32, 12288, False), "14b": (5120, 40, 40, 17408, False)}
DESIGNS = ("tezinex", "povatar", "pabavik", "pasovik", "kelisun", "puvirax")


# -------------------------------------------------------------------------------------------------- the cases
def case(name, design, size, requests, prompt, decode, ragged=False, dtype="bfloat16"):
    """requests prompts of `prompt` tokens (ragged: down to about a fifth of that), then `decode` steps of one token a request."""
    return {"name": name, "design": design, "size": size, "dtype": dtype, "requests": requests, "prompt": prompt, "ragged": ragged,
            "decode": decode}


def listed():
    return [
        # An interactive request to the smallest model: launches and latency are all there is.
        case("qwen3 0.6b short", "qwen3", "0.6b", 1, 23, 12),
        # The headline prompt: 2,048 tokens through the 8B shape.
        case("qwen3 8b prompt", "qwen3", "8b", 1, 2048, 0),
        # A chat batch on the 8B shape: eight prompts, then their decoding.
        case("qwen3 8b chat", "qwen3", "8b", 8, 512, 24),
        # Prompts of unequal lengths into the largest shape, more decoding rows than a tile of 16.
        case("qwen3 14b ragged", "qwen3", "14b", 19, 333, 5, ragged=True),
        # The 32-bit build, as it is used to check the other.
        case("qwen3 1.7b float32", "qwen3", "1.7b", 3, 217, 6, dtype="float32"),
        # Long prompts through the other designs at their largest size, each with its own mixers.
        case("tezinex 4k prompt", "tezinex", "4k", 1, 2048, 0),
        case("pabavik 4k prompt", "pabavik", "4k", 1, 2048, 0),
        case("pasovik 4k prompts", "pasovik", "4k", 3, 1111, 2, ragged=True),
        # Batches that generate: prompts and decoding in one pass.
        case("povatar 2k chat", "povatar", "2k", 8, 256, 16, ragged=True),
        case("kelisun 2k chat", "kelisun", "2k", 8, 300, 16),
        case("puvirax 4k chat", "puvirax", "4k", 5, 400, 12, ragged=True),
        # A short exchange with a small recurrent model.
        case("tezinex 1k short", "tezinex", "1k", 2, 150, 16),
    ]


def draw(rng):
    """One more case: any design and size, one to 24 requests, prompts of one to 2,048 tokens in all, up to 24 decoded tokens."""
    if rng.random() < 0.4:
        design, size = "qwen3", rng.choice(["0.6b", "1.7b", "4b", "8b"])
    else:
        design, size = rng.choice(DESIGNS), rng.choice(list(SIZES))
    requests = round(math.exp(rng.uniform(0.0, math.log(24))))
    prompt = max(1, round(math.exp(rng.uniform(math.log(4), math.log(2048))) / requests))
    dtype = "float32" if rng.random() < 0.15 and size in ("0.6b", "1.7b", "1k") else "bfloat16"
    out = case("", design, size, requests, prompt, rng.randrange(0, 25), rng.random() < 0.5, dtype)
    del out["name"]
    return out


def lengths(c):
    n = c["requests"]
    return [max(1, c["prompt"] - (i * c["prompt"] * 4) // (5 * n)) if c["ragged"] else c["prompt"] for i in range(n)]


# ------------------------------------------------------------------------------------------------ descriptions
def config_of(c):
    if c["design"] == "qwen3":
        width, layers, heads, ff, tied = QWEN3[c["size"]]
        return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "vocab_size": 151936, "hidden_size": width,
                "intermediate_size": ff, "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": 8, "head_dim": 128,
                "max_position_embeddings": 40960, "rms_norm_eps": 1e-6, "rope_theta": 1e6, "tie_word_embeddings": tied}
    width, heads, kv, ff = SIZES[c["size"]]
    sized = {"dim": 128, "vdim": 128, "heads": heads}
    attn = dict(sized, kv_heads=kv, scale=128 ** -0.5)
    base = {"architecture": c["design"].capitalize(), "norm": {"eps": 1e-5}, "vocab": VOCAB, "width": width}
    layers = []
    if c["design"] == "tezinex":
        mlp = {"kind": "dense", "ff": ff}
        for i in range(LAYERS):
            if i % 4 in (0, 3):
                layers.append({"type": "channel_delta", "mixer": dict(sized, kv_heads=heads, conv=4), "mlp": mlp})
            else:
                m = dict(attn, mask={"size": 1024, "keep_first": 16}, softcap=20.0)
                layers.append({"type": "attention", "mixer": dict(m, kv_from=i - 1) if i % 4 == 2 else m, "mlp": mlp})
        return dict(base, layers=layers, logit_softcap=20.0, residual_mult=0.5)
    if c["design"] == "povatar":
        left = dict(attn, mask={"size": 1024}, rot={"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "fast": 16.0, "original": 4096, "slow": 2.0}})
        right = {"conv": 4, "groups": 4, "heads": width // 64, "norm_groups": 4, "state": 128, "vdim": 64}
        mlp = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 32, "top": 4}}
        return dict(base, embedding={"scale": 1.0}, layers=[{"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": mlp}] * LAYERS)
    if c["design"] == "pabavik":
        mlp = {"kind": "moe", "expert": {"ff": ff // 4, "limit": 7.0}, "router": {"experts": 32, "top": 3}, "shared": {"ff": ff // 4, "limit": 7.0}}
        for i in range(LAYERS):
            if i % 4 in (0, 3):
                layers.append({"type": "gla", "mixer": dict(sized, tau=16.0), "mlp": mlp})
            else:
                m = dict(attn, mask={"size": 1024}, rot={"base": 10000.0, "dims": 64})
                layers.append({"type": "attention", "mixer": dict(m, kv_from=i - 1) if i % 4 == 2 else m, "mlp": mlp})
        return dict(base, embedding={"scale": 1.0}, layers=layers, logit_softcap=20.0)
    if c["design"] == "pasovik":
        dense = {"kind": "dense", "ff": ff}
        moe = {"kind": "moe", "expert": {"ff": ff // 4, "limit": 7.0}, "router": {"experts": 32, "top": 4}}
        decay = [1.0 - 2.0 ** (-5.0 - 5.0 * h / max(heads - 1, 1)) for h in range(heads)]
        latent = dict(sized, rot_dim=64, kv_rank=192, q_rank=width // 2, scale=192 ** -0.5, rot={"base": 10000.0, "dims": 64})
        for i in range(LAYERS):
            layers.append([{"type": "lightning", "mixer": dict(sized, decay=decay), "mlp": dense},
                           {"type": "attention", "mixer": dict(attn, softcap=30.0, rot={"base": 10000.0, "dims": 64, "scaling": {"factor": 8.0}}), "mlp": moe},
                           {"type": "latent_attention", "mixer": latent, "mlp": dense},
                           {"type": "latent_attention", "mixer": dict(latent, kv_from=i - 1), "mlp": moe}][i % 4])
        return dict(base, layers=layers, token_side={"dim": 256})
    if c["design"] == "kelisun":
        mlp = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 32, "top": 4, "groups": {"count": 8, "keep": 4}, "scale": 2.5}}
        for i in range(LAYERS):
            m = dict(sized, rot_dim=64, kv_rank=192, scale=192 ** -0.5, mask={"size": 1024 if i % 2 == 0 else 1536},
                     rot={"base": 10000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 2048, "fast": 16.0, "slow": 1.0}})
            layers.append(dict(layers[i - 1], weights_of=i - 1) if i % 4 == 3 else {"type": "latent_attention", "mixer": m, "mlp": mlp})
        return dict(base, layers=layers, streams=4)
    dense = {"kind": "dense", "ff": 3 * ff // 2}
    moe = {"kind": "moe", "expert": {"ff": 3 * ff // 8}, "router": {"experts": 32, "top": 3, "groups": {"count": 8, "keep": 4}}, "shared": {"ff": 3 * ff // 8}}
    attn = dict(attn, v_mix=True)
    kinds = [("attention_2", dict(attn, bias_max=128, mask={"size": 1024})), ("attention_3", dict(attn, bias_max=128))]
    kinds += [("attention", dict(attn, rot={"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 2048}}))] * 2
    layers = [{"type": kinds[i % 4][0], "mixer": kinds[i % 4][1], "mlp": moe if i % 2 else dense} for i in range(LAYERS)]
    return dict(base, embedding={"bigram": {"buckets": VOCAB - 3, "mul_cur": 29, "mul_prev": 13}}, layers=layers, logit_scale=0.25)


def tensors_of(c):
    """Every stored tensor: name -> (shape, standard deviation, or the bounds of a uniform draw)."""
    cfg, t = config_of(c), {}
    near_one, near_zero = (0.9, 1.1), (-0.1, 0.1)
    if c["design"] == "qwen3":
        H, nq, nkv, d, ff, V = cfg["hidden_size"], cfg["num_attention_heads"], 8, 128, cfg["intermediate_size"], cfg["vocab_size"]
        t["model.embed_tokens.weight"] = ((V, H), 0.02)
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            for n in ("input_layernorm", "post_attention_layernorm"):
                t[p + n + ".weight"] = ((H,), near_one)
            t.update({p + f"self_attn.{n}_norm.weight": ((d,), near_one) for n in "qk"})
            t.update({p + f"self_attn.{n}_proj.weight": ((k * d, H), 0.02) for n, k in (("q", nq), ("k", nkv), ("v", nkv))})
            t[p + "self_attn.o_proj.weight"] = ((H, nq * d), 0.02)
            t.update({p + f"mlp.{n}_proj.weight": ((ff, H), 0.02) for n in ("gate", "up")})
            t[p + "mlp.down_proj.weight"] = ((H, ff), 0.02)
        t["model.norm.weight"] = ((H,), near_one)
        if not cfg["tie_word_embeddings"]:
            t["lm_head.weight"] = ((V, H), 0.02)
        return t
    W, V, design = cfg["width"], cfg["vocab"], c["design"]
    norms = near_zero if design in ("tezinex", "pabavik") else near_one
    rank = max(8, W // 16)

    def attention(p, m, kind="attention"):
        H, d = m["heads"], m["dim"]
        G = m.get("kv_heads", H)
        own = m.get("kv_from") is None
        t[p + "q"] = ((H * d, W), 0.02)
        if own:
            t[p + "k"] = t[p + "v"] = ((G * d, W), 0.02)
        t[p + "o"] = ((W, H * d), 0.02)
        if design == "tezinex":
            t[p + "q.b"], t[p + "sink"] = ((H * d,), 0.02), ((H,), (-1.0, 1.0))
            if own:
                t[p + "k.b"] = t[p + "v.b"] = ((G * d,), 0.02)
        if design == "pabavik":
            t[p + "g"] = ((H * d, W), 0.02)
        if design in ("pabavik", "pasovik") or kind == "attention_2":
            t[p + "q.norm"] = ((d,), near_one)
            if own:
                t[p + "k.norm"] = ((d,), near_one)
        if kind == "attention_3":
            t[p + "q.norm"], t[p + "k.norm"] = ((H * d,), near_one), ((G * d,), near_one)
        if kind in ("attention_2", "attention_3"):
            t[p + "rel"] = ((32, H), 1.0)
        if design == "puvirax" and kind == "attention":
            t[p + "g"] = ((H, W), 0.02)

    def matrices(p, m):
        ups = ("up",) if design in ("povatar", "puvirax") else ("gate", "up")
        t.update({p + n: ((m["ff"], W), 0.02) for n in ups})
        t[p + "down"] = ((W, m["ff"]), 0.02)

    t["embed"] = ((V, W), 0.02)
    for i, layer in enumerate(cfg["layers"]):
        if layer.get("weights_of") is not None:
            continue
        p, m, kind = f"l{i}.", layer["mixer"], layer["type"]
        x = p + "mix."
        for n in {"tezinex": ("norm1", "norm1b", "norm2", "norm2b"), "pabavik": ("norm1", "norm1b", "norm2", "norm2b")}.get(design, ("norm1", "norm2")):
            t[p + n] = ((W,), norms)
        H, d = m.get("heads"), m.get("dim")
        if kind == "parallel":
            attention(x + "left.", m["left"])
            r, y = m["right"], x + "right."
            inner, channels = r["heads"] * r["vdim"], r["heads"] * r["vdim"] + 2 * r["groups"] * r["state"]
            t.update({y + "in": ((inner + channels + r["heads"], W), 0.05), y + "conv": ((channels, r["conv"]), 0.3), y + "conv.b": ((channels,), (-0.1, 0.1)),
                      y + "dt_bias": ((r["heads"],), (-2.0, 0.0)), y + "A_log": ((r["heads"],), (-1.0, 1.0)), y + "D": ((r["heads"],), (0.5, 1.5)),
                      y + "norm": ((inner,), near_one), y + "o": ((W, inner), 0.02), x + "left.out": ((W,), near_one), y + "out": ((W,), near_one)})
        elif kind == "channel_delta":
            t.update({x + n: ((H * d, W), 0.1) for n in "qkv"})
            t.update({x + n + ".conv": ((H * d, m["conv"]), 0.3) for n in "qkv"})
            t.update({x + "b": ((H, W), 0.02), x + "A_log": ((H,), (-1.0, 1.0)), x + "norm": ((d,), near_one), x + "a1": ((rank, W), 0.02),
                      x + "a2": ((H * d, rank), 0.02), x + "dt_bias": ((H * d,), (-1.0, 1.0)), x + "g1": ((rank, W), 0.02),
                      x + "g2": ((H * d, rank), 0.02), x + "o": ((W, H * d), 0.02)})
        elif kind in ("gla", "lightning"):
            t.update({x + n: ((H * d, W), 0.1) for n in "qkv"})
            t.update({x + "g": ((H * d, W), 0.02), x + "o": ((W, H * d), 0.02), x + "norm": ((d if kind == "gla" else H * d,), near_one)})
            if kind == "gla":
                t.update({x + "a1": ((rank, W), 0.02), x + "a2": ((H * d, rank), 0.5), x + "a2.b": ((H * d,), (1.0, 5.0))})
        elif kind == "latent_attention":
            dr, r, rq = m["rot_dim"], m["kv_rank"], m.get("q_rank")
            t.update({x + "uk": ((H * d, r), 0.06), x + "uv": ((H * d, r), 0.06), x + "o": ((W, H * d), 0.02)})
            if rq:
                t.update({x + "dq": ((rq, W), 0.02), x + "dq.norm": ((rq,), near_one), x + "uq": ((H * (d + dr), rq), 0.06), x + "g": ((H * d, W), 0.02)})
            else:
                t.update({x + "q": ((H * (d + dr), W), 0.02), x + "sink": ((H,), (-1.0, 1.0))})
            if m.get("kv_from") is None:
                t.update({x + "dkv": ((r + dr, W), 0.02), x + "dkv.norm": ((r,), near_one)})
        else:
            attention(x, m, kind)
            if m.get("v_mix") and i > 0:
                t[x + "vmix"] = ((), (0.3, 0.7))
        mlp, x = layer["mlp"], p + "mlp."
        if mlp["kind"] == "dense":
            matrices(x, mlp)
        else:
            t[x + "router"] = ((mlp["router"]["experts"], W), 0.1)
            for n in {"pabavik": ("router.b",), "puvirax": ("correction",)}.get(design, ()):
                t[x + n] = ((mlp["router"]["experts"],), (-0.5, 0.5))
            for e in range(mlp["router"]["experts"]):
                matrices(f"{x}e{e}.", mlp["expert"])
            if mlp.get("shared"):
                matrices(x + "shared.", mlp["shared"])
        if design == "tezinex":
            t[p + "dwa"] = ((i + 2,), (0.0, 2.0 / (i + 2)))
        if design == "pasovik":
            t.update({p + "side.gate": ((256, W), 0.05), p + "side.proj": ((W, 256), 0.2), p + "side.norm": ((W,), near_one)})
        if design == "kelisun":
            for n in ("hc1.", "hc2."):
                t.update({p + n + "in": ((4,), (0.5, 1.0)), p + n + "out": ((4,), (0.7, 1.3)), p + n + "mix": ((4, 4), (0.125, 0.375))})
    t["final.norm"] = ((W,), norms)
    if design not in ("tezinex", "puvirax"):
        t["head"] = ((V, W), 0.02)
    if design == "pasovik":
        t["side.embed"] = ((V, 256 * LAYERS), 1.0)
    if design == "kelisun":
        t["embed.norm"] = ((W,), near_one)
    if design == "puvirax":
        t["bigram"] = ((VOCAB - 2, W), 0.02)
    return t


# ---------------------------------------------------------------------------------------------------- the pass
def token_ids(c, seed):
    """The tokens of every request, prompt and continuation."""
    rng = np.random.default_rng([seed, 77])
    vocab = config_of(c).get("vocab_size", VOCAB)
    return [rng.integers(0, vocab, n + c["decode"]).tolist() for n in lengths(c)]


def steps_of(c, tokens):
    """What is fed to the engine step by step: entries (request, its next tokens, wanted places among them)."""
    ends = list(enumerate(lengths(c)))
    steps = [[(r, tokens[r][:n], [n - 1]) for r, n in ends]]
    return steps + [[(r, [tokens[r][n + k]], [0]) for r, n in ends] for k in range(c["decode"])]


def prepare(c, seed):
    from vosti_amd.engine import create_engine
    pages = sum(-(-(n + c["decode"] + 1) // PAGE) for n in lengths(c)) + 2
    with tempfile.TemporaryDirectory() as folder:
        (Path(folder) / "config.json").write_text(json.dumps(config_of(c)))
        engine = create_engine(folder, dtype=c["dtype"], random_weights_seed=seed, num_pages=pages, page_size=PAGE, max_num_seqs=c["requests"],
                               max_num_batched_tokens=STEP_TOKENS, enable_prefix_cache=False, graphs=True)
    return {"engine": engine, "steps": steps_of(c, token_ids(c, seed)), "requests": c["requests"]}


def run(state):
    engine = state["engine"]
    logits = [engine.trace_step(entries) for entries in state["steps"]]
    for r in range(state["requests"]):
        engine.trace_finish(r)
    return logits


def attention_span(c, layer):
    """Keys that a row of this layer's attention sees at most (0: the layer has none)."""
    if layer["type"] in ("channel_delta", "gla", "lightning"):
        return 0
    m = layer["mixer"].get("left", layer["mixer"])
    return (m.get("mask") or {}).get("size", 1 << 30)


def work(c):
    """Weights once a step (of the experts, those that the step's tokens can be expected to choose), every visible key and value once a
    step and request, states read and written, logits out; two operations a weight and token, four a visible (row, key, entry)."""
    cfg, elem = config_of(c), 4 if c["dtype"] == "float32" else 2
    layers = cfg.get("layers", [])
    router = next((x["mlp"]["router"] for x in layers if x["mlp"]["kind"] == "moe"), None)
    share = router["top"] / router["experts"] if router else 0.0
    dense = expert = 0
    for name, (shape, _) in tensors_of(c).items():
        n = math.prod(shape)
        if ".mlp.e" in name:
            expert += n
        elif not (name.endswith("embed") or "embed_tokens" in name or name == "bigram"):
            dense += n
    vocab, width = cfg.get("vocab_size", VOCAB), cfg.get("hidden_size", cfg.get("width"))
    head = vocab * width
    dense -= head if ("head" in tensors_of(c) or "lm_head.weight" in tensors_of(c)) else 0
    if c["design"] == "qwen3":
        spans = [(1 << 30, 2 * 8 * 128, cfg["num_attention_heads"], 128)] * cfg["num_hidden_layers"]
        state = 0
    else:
        spans, state = [], 0
        for x in layers:
            m = x["mixer"].get("left", x["mixer"])
            latent = x["type"] == "latent_attention"
            if attention_span(c, x):
                spans.append((attention_span(c, x), 256 if latent else 2 * m["kv_heads"] * 128, m["heads"], 256 if latent else 128))
            if x["type"] == "parallel":
                state += x["mixer"]["right"]["heads"] * 64 * 128 * 4
            elif not attention_span(c, x):
                state += m["heads"] * 128 * 128 * 4
    nbytes = flops = 0.0
    for step in steps_of(c, [[0] * (n + c["decode"]) for n in lengths(c)]):
        rows = sum(len(e[1]) for e in step)
        wanted = sum(len(e[2]) for e in step)
        nbytes += elem * (dense + head + expert * (1.0 - (1.0 - share) ** rows)) + 4.0 * wanted * vocab + elem * rows * width
        flops += 2.0 * rows * (dense + share * expert) + 2.0 * wanted * head
        nbytes += 2.0 * state * len(step)
    done = 0
    for n in lengths(c):
        for span, kept, heads, d in spans:
            sees = [min(span, p + 1) for p in range(n + c["decode"])]
            flops += 4.0 * heads * d * sum(sees)
            nbytes += elem * kept * (min(span, n) + sum(sees[n:]))
        done += n
    return {"bytes": nbytes, "flops": flops}


def routed(c):
    return c["design"] not in ("qwen3", "tezinex")


def tolerance(c):
    """The 2-norm of the difference over all logits of a pass, about four times what `exact` shows where there is one: 32-bit 2e-5 at most
    without a router and 4e-5 behind recurrences over a thousand tokens; bfloat16 0.004 in eight layers and 0.056 in forty.  In bfloat16
    a router whose best candidates all but tie chooses another expert when a sum's last bit changes, and the row behind it differs
    by 0.1 to 0.6."""
    if c["dtype"] == "float32":
        return {"rel": 1e-4}
    if routed(c):
        return {"rel": 0.6}
    return {"rel": 0.2 if c["design"] == "qwen3" else 0.016}


# --------------------------------------------------------------------------------------- the same in 64 bits
F64 = torch.float64


class Weights:
    """w[name]: the values that the model holds, as 64-bit numbers.  Element i of a tensor is a function of (seed, name, i): the
    counter i * golden, xored with the first 8 bytes of BLAKE2b("seed:name"), through the finaliser of splitmix64; a normal value is
    the sum of its four 16-bit pieces, centred and scaled, a uniform one its upper 24 bits."""

    def __init__(self, c, seed):
        self.tensors, self.seed = tensors_of(c), seed
        self.dtype = getattr(torch, c["dtype"])

    def __contains__(self, name):
        return name in self.tensors

    def __getitem__(self, name):
        shape, init = self.tensors[name]
        n = math.prod(shape)
        out = torch.empty(n, dtype=F64, device="cuda")
        key = int.from_bytes(hashlib.blake2b(f"{self.seed}:{name}".encode(), digest_size=8).digest(), "little", signed=True)

        def signed(v):
            return v - (1 << 64) if v >= 1 << 63 else v

        def down(z, bits):                       # a logical shift
            return (z >> bits) & ((1 << (64 - bits)) - 1)
        for a in range(0, n, 1 << 25):
            z = torch.arange(a, min(n, a + (1 << 25)), device="cuda") * signed(0x9E3779B97F4A7C15) ^ key
            z = (z ^ down(z, 30)) * signed(0xBF58476D1CE4E5B9)
            z = (z ^ down(z, 27)) * signed(0x94D049BB133111EB)
            z = z ^ down(z, 31)
            if isinstance(init, tuple):
                u = down(z, 40).to(torch.float32) * 2.0 ** -24
                v = u * float(np.float32(init[1] - init[0])) + float(np.float32(init[0]))
            else:
                total = (z & 0xFFFF) + (down(z, 16) & 0xFFFF) + (down(z, 32) & 0xFFFF) + down(z, 48) - 131070
                v = total.to(torch.float32) * float(np.float32(init * math.sqrt(3.0) / 65536.0))
            out[a:a + len(v)] = v.to(self.dtype).to(F64)
        return out.view(shape)


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(z):
    return z * torch.sigmoid(z)


def frequencies(rot, design):
    dims = rot["dims"]
    i = torch.arange(dims // 2, dtype=F64, device="cuda")
    f = rot["base"] ** (-2.0 * i / dims)
    sc = rot.get("scaling")
    if not sc:
        return f, 1.0
    if design == "pasovik":
        return f / sc["factor"], 1.0
    if design == "puvirax":                      # by wavelength: short ones stay, long ones are divided, a blend between
        turns = sc["original"] * f / (2.0 * math.pi)
        s = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        return (1.0 - s) * f / sc["factor"] + s * f, 1.0

    def index_of(turns):
        return dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))
    low, high = max(math.floor(index_of(sc["fast"])), 0), min(math.ceil(index_of(sc["slow"])), dims - 1)
    ramp = ((i - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
    return f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def rotate(x, rot, design):
    """x [T, heads, d] from position 0: the first dims entries in pairs of halves (pasovik: of neighbours)."""
    dims = rot["dims"]
    f, mag = frequencies(rot, design)
    angle = torch.arange(len(x), dtype=F64, device="cuda")[:, None, None] * f
    cos, sin = torch.cos(angle) * mag, torch.sin(angle) * mag
    first, second = (slice(0, dims, 2), slice(1, dims, 2)) if design == "pasovik" else (slice(0, dims // 2), slice(dims // 2, dims))
    u, v, out = x[..., first], x[..., second], x.clone()
    out[..., first], out[..., second] = u * cos - v * sin, v * cos + u * sin
    return out


def attend(q, k, v, scale, see=None, softcap=None, sink=None, bias=None):
    """q [T, H, d], k and v [T, G, .]; see(i, j) what is visible beside causality; sink: a number a head as one more score."""
    T, H, G = len(q), q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=F64, device="cuda")
    j = torch.arange(T, device="cuda")
    back = j[:, None] - j[None, :]
    hidden = back < 0
    if see is not None:
        hidden |= ~see(j[:, None], j[None, :])
    for h in range(H):
        s = q[:, h] @ k[:, h * G // H].T * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        if bias is not None:
            s = s + bias[back.clamp(min=0), h]
        s = s.masked_fill(hidden, -math.inf)
        top = s.amax(1, keepdim=True)
        top = top if sink is None else top.clamp(min=float(sink[h]))
        e = torch.exp(s - top)
        total = e.sum(1, keepdim=True) + (0.0 if sink is None else torch.exp(sink[h] - top))
        out[:, h] = e @ v[:, h * G // H] / total
    return out


def scan(decay, k, v, q, beta=None):
    """S <- decay S + k (x) v (with beta: v is beta (v - S^T k)), o = S^T q, token by token.  All [T, H, .]."""
    T, H, d = k.shape
    S = torch.zeros(H, d, v.shape[2], dtype=F64, device="cuda")
    out = torch.empty(T, H, v.shape[2], dtype=F64, device="cuda")
    for t in range(T):
        S = decay[t][:, :, None] * S
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        out[t] = (S * q[t][:, :, None]).sum(1)
    return out


def conv(x, taps, bias=0.0):
    T, K = len(x), taps.shape[1]
    x = torch.cat([torch.zeros(K - 1, x.shape[1], dtype=F64, device="cuda"), x])
    return sum(x[j:j + T] * taps[:, j] for j in range(K)) + bias


def each(parts, f, *rows):
    """f on every sequence of the rows, side by side again."""
    return torch.cat([f(*(r[a:b] for r in rows)) for a, b in parts])


def heads(x, n):
    return x.view(len(x), n, -1)


def feed_forward(w, p, h, design, limit=None):
    up = h @ w[p + "up"].T
    if design in ("povatar", "puvirax"):
        return torch.relu(up) ** 2 @ w[p + "down"].T
    gate = h @ w[p + "gate"].T
    if limit is None:
        return silu(gate) * up @ w[p + "down"].T
    gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
    return gate * torch.sigmoid(1.702 * gate) * (up + 1.0) @ w[p + "down"].T


def experts(w, p, h, mlp, design):
    router = mlp["router"]
    z, top = h @ w[p + "router"].T, router["top"]
    score = torch.sigmoid(z) if design in ("pasovik", "puvirax") else torch.softmax(z, -1)
    if design == "pasovik":                      # scores of 32 bits reach 1, and the first of those that do are chosen
        score = torch.sigmoid(z.float()).to(F64)
    choice = z + w[p + "router.b"] if design == "pabavik" else score + w[p + "correction"] if design == "puvirax" else score
    if router.get("groups"):
        g = choice.view(len(h), router["groups"]["count"], -1)
        worth = g.topk(2, -1).values.sum(-1) if design == "puvirax" else g.amax(-1)
        kept = torch.zeros_like(worth, dtype=torch.bool).scatter(1, worth.topk(router["groups"]["keep"], -1).indices, True)
        allowed = g.masked_fill(~kept[:, :, None], -math.inf).view_as(choice)
    else:
        allowed = choice
    idx = torch.sort(allowed, dim=-1, descending=True, stable=True).indices[:, :top]
    weight = torch.softmax(choice.gather(1, idx), -1) if design == "pabavik" else score.gather(1, idx) * router.get("scale", 1.0)
    if design == "povatar":
        weight = weight / weight.sum(-1, keepdim=True)
    limit = mlp["expert"].get("limit")
    out = feed_forward(w, p + "shared.", h, design, limit) if mlp.get("shared") else torch.zeros_like(h)
    for e in range(router["experts"]):
        rows, place = (idx == e).nonzero(as_tuple=True)
        by = weight[rows, place][:, None]
        if design == "pasovik":                  # the score scales what the expert reads
            out[rows] += feed_forward(w, f"{p}e{e}.", by * h[rows], design, limit)
        else:
            out[rows] += by * feed_forward(w, f"{p}e{e}.", h[rows], design, limit)
    return out


def mixer(w, p, h, layer, design, eps, parts, kept, i, shared):
    """A layer's mixer on rows of several sequences.  kept: keys and values that later layers read; shared: the first layer's values."""
    m, kind = layer["mixer"], layer["type"]
    if kind == "parallel":
        left = mixer(w, p + "left.", h, {"type": "attention", "mixer": m["left"]}, design, eps, parts, kept, i, shared)
        right = mixer(w, p + "right.", h, {"type": "state_space", "mixer": m["right"]}, design, eps, parts, kept, i, shared)
        return 0.5 * (rms(left, eps) * w[p + "left.out"] + rms(right, eps) * w[p + "right.out"])
    H = m["heads"]
    if kind == "state_space":
        P, N, G = m["vdim"], m["state"], m["groups"]
        z, xbc, dt = (h @ w[p + "in"].T).split([H * P, H * P + 2 * G * N, H], 1)
        taps, bias = w[p + "conv"], w[p + "conv.b"]
        x, B, C = silu(each(parts, lambda r: conv(r, taps, bias), xbc)).split([H * P, G * N, G * N], 1)
        dt = torch.nn.functional.softplus(dt + w[p + "dt_bias"])
        decay = torch.exp(-torch.exp(w[p + "A_log"]) * dt)[:, :, None].expand(-1, -1, N)
        x, B, C = heads(x, H), heads(B, G).repeat_interleave(H // G, 1), heads(C, G).repeat_interleave(H // G, 1)
        y = each(parts, scan, decay, B, dt[:, :, None] * x, C) + w[p + "D"][:, None] * x
        y = rms(heads(y.reshape(len(h), -1) * silu(z), m["norm_groups"]), eps).reshape(len(h), -1)
        return y * w[p + "norm"] @ w[p + "o"].T
    if kind == "channel_delta":
        def taken(n):
            taps = w[p + n + ".conv"]
            return heads(silu(each(parts, lambda r: conv(r, taps), h @ w[p + n].T)), H)
        q, k, v = taken("q"), taken("k"), taken("v")
        q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * m["dim"] ** -0.5
        k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        a = heads(h @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "dt_bias"], H)
        decay = torch.exp(-torch.exp(w[p + "A_log"])[:, None] * torch.nn.functional.softplus(a))
        o = each(parts, scan, decay, k, v, q, torch.sigmoid(h @ w[p + "b"].T))
        o = rms(o, eps) * w[p + "norm"] * heads(torch.sigmoid(h @ w[p + "g1"].T @ w[p + "g2"].T), H)
        return o.reshape(len(h), -1) @ w[p + "o"].T
    if kind in ("gla", "lightning"):
        q, k, v = (heads(h @ w[p + n].T, H) for n in "qkv")
        gate = h @ w[p + "g"].T
        if kind == "gla":
            z = h @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "a2.b"]
            decay = heads(torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]), H)
            o = rms(each(parts, scan, decay, k, v, q * m["dim"] ** -0.5), eps) * w[p + "norm"]
            return o.reshape(len(h), -1) * silu(gate) @ w[p + "o"].T
        decay = torch.tensor(m["decay"], dtype=F64, device="cuda")[None, :, None].expand(len(h), -1, m["dim"])
        o = each(parts, scan, decay, silu(k), silu(v), silu(q)).reshape(len(h), -1)
        return rms(o, eps) * w[p + "norm"] * torch.sigmoid(gate) @ w[p + "o"].T
    size = (m.get("mask") or {}).get("size")
    if kind == "latent_attention":
        d, r = m["dim"], m["kv_rank"]
        q = heads(rms(h @ w[p + "dq"].T, eps) * w[p + "dq.norm"] @ w[p + "uq"].T if m.get("q_rank") else h @ w[p + "q"].T, H)
        if m.get("kv_from") is None:
            down = h @ w[p + "dkv"].T
            kept[i] = rms(down[:, :r], eps) * w[p + "dkv.norm"], each(parts, lambda x: rotate(x, m["rot"], design), down[:, None, r:])
        else:
            kept[i] = kept[m["kv_from"]]
        c, turned = kept[i]
        q = torch.cat([q[..., :d], each(parts, lambda x: rotate(x, m["rot"], design), q[..., d:])], -1)
        k = torch.cat([heads(c @ w[p + "uk"].T, H), turned.expand(-1, H, -1)], -1)
        v = heads(c @ w[p + "uv"].T, H)
        sink = w[p + "sink"] if p + "sink" in w else None
        see = (lambda a, b: a - b < size) if size else None
        o = each(parts, lambda a, b, x: attend(a, b, x, m["scale"], see, sink=sink), q, k, v).reshape(len(h), -1)
        return (o * torch.sigmoid(h @ w[p + "g"].T) if p + "g" in w else o) @ w[p + "o"].T
    G = m["kv_heads"]
    own = m.get("kv_from") is None
    plus = (lambda n: w[p + n + ".b"]) if design == "tezinex" else (lambda n: 0.0)
    q = heads(h @ w[p + "q"].T + plus("q"), H)
    if own:
        k, v = heads(h @ w[p + "k"].T + plus("k"), G), heads(h @ w[p + "v"].T + plus("v"), G)

    def placed(x, n):                            # norms and rotation of queries or keys, in the design's order
        if kind == "attention_3":
            return heads(rms(x.flatten(1), eps) * w[p + n + ".norm"], x.shape[1])
        if p + n + ".norm" in w:
            x = rms(x, eps) * w[p + n + ".norm"]
        if m.get("rot"):
            x = each(parts, lambda r: rotate(r, m["rot"], design), x)
        return rms(x, eps) if design == "puvirax" and kind == "attention" else x
    q = placed(q, "q")
    if own:
        if m.get("v_mix"):
            v = (1.0 - w[p + "vmix"]) * v + w[p + "vmix"] * shared["v"] if "v" in shared else shared.setdefault("v", v)
        kept[i] = placed(k, "k"), v
    else:
        kept[i] = kept[m["kv_from"]]
    k, v = kept[i]
    sink = bias = see = None
    if design == "tezinex":
        keep = m["mask"]["keep_first"]
        sink, see = w[p + "sink"], lambda a, b: (a - b < size) | (b < keep)
    elif design == "povatar":
        sink, see = torch.zeros(H, dtype=F64, device="cuda"), lambda a, b: a // size == b // size
    elif size:
        sink, see = torch.zeros(H, dtype=F64, device="cuda") if design == "pabavik" else None, lambda a, b: a - b < size
    if p + "rel" in w:
        rows, far = w[p + "rel"].shape[0], m["bias_max"]
        half = rows // 2
        classes = [n if n < half else min(rows - 1, half + math.floor(math.log(n / half) / math.log(far / half) * (rows - half)))
                   for n in range(max(b - a for a, b in parts))]
        bias = w[p + "rel"][torch.tensor(classes, device="cuda")]
    o = each(parts, lambda a, b, x: attend(a, b, x, m["scale"], see, m.get("softcap"), sink, bias), q, k, v)
    if design == "puvirax" and kind == "attention":
        o = o * torch.sigmoid(h @ w[p + "g"].T)[:, :, None]
    o = o.reshape(len(h), -1)
    return (o * torch.sigmoid(h @ w[p + "g"].T) if design == "pabavik" else o) @ w[p + "o"].T


def design_logits(c, w, tokens, parts, wanted):
    cfg, design = config_of(c), c["design"]
    eps = cfg["norm"]["eps"]
    offset = 1.0 if design in ("tezinex", "pabavik") else 0.0
    flat = torch.tensor([t for s in tokens for t in s], device="cuda")

    def norm(x, name):
        return rms(x, eps) * (offset + w[name])

    def output(x, p, layer):
        return experts(w, p, x, layer["mlp"], design) if layer["mlp"]["kind"] == "moe" else feed_forward(w, p, x, design)
    x = w["embed"][flat]
    if design == "tezinex":
        half = torch.arange(cfg["width"] // 2, dtype=F64, device="cuda")
        place = torch.cat([torch.arange(b - a, dtype=F64, device="cuda") for a, b in parts])
        angle = place[:, None] * 10000.0 ** (-2.0 * half / cfg["width"])
        x = x + torch.stack([torch.sin(angle), torch.cos(angle)], -1).flatten(1)
    if design == "puvirax":
        b = cfg["embedding"]["bigram"]
        rows = [b["buckets"] if k == 0 else (s[k - 1] * b["mul_prev"] + t * b["mul_cur"]) % b["buckets"] for s in tokens for k, t in enumerate(s)]
        x = x + w["bigram"][torch.tensor(rows, device="cuda")]
    if design == "kelisun":
        x = norm(x, "embed.norm")[None].repeat(4, 1, 1)
    kept, shared, results = {}, {}, [x]
    for i, layer in enumerate(cfg["layers"]):
        p = f"l{i if layer.get('weights_of') is None else layer['weights_of']}."

        def mixed(h):
            return mixer(w, p + "mix.", h, layer, design, eps, parts, kept, i, shared)
        if design == "tezinex":
            x = x + cfg["residual_mult"] * norm(mixed(norm(x, p + "norm1")), p + "norm1b")
            x = x + cfg["residual_mult"] * norm(output(norm(x, p + "norm2"), p + "mlp.", layer), p + "norm2b")
            results.append(x)
            x = sum(a * b for a, b in zip(w[p + "dwa"], results))
        elif design == "povatar":
            x = x + mixed(norm(x, p + "norm1")) + output(norm(x, p + "norm2"), p + "mlp.", layer)
        elif design == "pabavik":
            x = x + norm(mixed(norm(x, p + "norm1")), p + "norm1b")
            x = x + norm(output(norm(x, p + "norm2"), p + "mlp.", layer), p + "norm2b")
        elif design == "pasovik":
            x = x + norm(mixed(x), p + "norm1")
            x = x + norm(output(x, p + "mlp.", layer), p + "norm2")
            side = w["side.embed"][flat, i * 256:(i + 1) * 256] * torch.nn.functional.gelu(x @ w[p + "side.gate"].T, approximate="tanh")
            x = x + norm(side @ w[p + "side.proj"].T, p + "side.norm")
        elif design == "kelisun":
            for n, f in (("1", mixed), ("2", lambda h: output(h, p + "mlp.", layer))):
                y = f(norm(torch.tensordot(w[p + f"hc{n}.in"], x, 1), p + "norm" + n))
                x = torch.tensordot(w[p + f"hc{n}.mix"].T, x, 1) + w[p + f"hc{n}.out"][:, None, None] * y
        else:
            x = x + mixed(norm(x, p + "norm1"))
            x = x + output(norm(x, p + "norm2"), p + "mlp.", layer)
    x = norm(x.sum(0) if design == "kelisun" else x, "final.norm")[wanted]
    logits = x @ w["head" if "head" in w else "embed"].T * cfg.get("logit_scale", 1.0)
    cap = cfg.get("logit_softcap")
    return cap * torch.tanh(logits / cap) if cap else logits


def qwen3_logits(c, w, tokens, parts, wanted):
    cfg = config_of(c)
    eps, nq = cfg["rms_norm_eps"], cfg["num_attention_heads"]
    rot = {"base": cfg["rope_theta"], "dims": 128}
    x = w["model.embed_tokens.weight"][torch.tensor([t for s in tokens for t in s], device="cuda")]
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = rms(x, eps) * w[p + "input_layernorm.weight"]
        a = p + "self_attn."
        q, k, v = (heads(h @ w[a + n + "_proj.weight"].T, nq if n == "q" else 8) for n in "qkv")
        q, k = (each(parts, lambda r: rotate(r, rot, "qwen3"), rms(r, eps) * w[a + n + "_norm.weight"]) for n, r in (("q", q), ("k", k)))
        o = each(parts, lambda s, t, u: attend(s, t, u, 128 ** -0.5), q, k, v)
        x = x + o.reshape(len(x), -1) @ w[a + "o_proj.weight"].T
        h = rms(x, eps) * w[p + "post_attention_layernorm.weight"]
        x = x + silu(h @ w[p + "mlp.gate_proj.weight"].T) * (h @ w[p + "mlp.up_proj.weight"].T) @ w[p + "mlp.down_proj.weight"].T
    x = (rms(x, eps) * w["model.norm.weight"])[wanted]
    return x @ w["lm_head.weight" if "lm_head.weight" in w else "model.embed_tokens.weight"].T


def exact(c, seed):
    """None where bfloat16 meets a router: which of two all but equal experts a row goes to has no value that 64 bits would tell."""
    if c["dtype"] == "bfloat16" and routed(c):
        return None
    tokens = token_ids(c, seed)
    parts, wanted, at = [], [], 0
    for s, n in zip(tokens, lengths(c)):
        parts.append((at, at + len(s)))
        wanted.append(list(range(at + n - 1, at + len(s))))
        at += len(s)
    rows = torch.tensor(wanted, device="cuda")                     # [request, wanted place]
    logits = (qwen3_logits if c["design"] == "qwen3" else design_logits)(c, Weights(c, seed), tokens, parts, rows.T.reshape(-1))
    return list(logits.view(rows.shape[1], len(tokens), -1).cpu().numpy())
