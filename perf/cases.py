"""The work this engine is measured by: whole requests through `Engine.add_request` and `Engine.step`, prompts and
generated tokens together, at the sizes of this repository's benchmark.

A pass hands a batch of prompts to a live engine, steps it until every request has its tokens and asks for the logits
behind the last of them.  What comes back are all generated tokens and these logits.  `prepare` keeps what a serving program keeps: the engine
with its weights, its steps captured for the shapes of this workload.

Weights are drawn here (the same in every process).  They are made so that a generation can be compared between two
implementations at all: the residual stream keeps the token's own embedding in view, as trained models' streams do,
and the output head's rows are the embedding's in another order, so the likeliest next token is far ahead of the
others, and a rounding error changes logits but not the sequence.  Queries and keys are scaled so that attention is
far from uniform, decays and gates lie where trained ones do.
"""
import math
import random
import zlib
from collections import OrderedDict

import torch

from tiny_llm_amd import Engine, SamplingParams, StepEntry
from tiny_llm_amd.weights import Checkpoint, load_weights

VOCAB = 32000
DEVICE = "cuda:0"


# ------------------------------------------------------------------------------------------------- the models
def llama(layers, width, heads, kv_heads, ff, vocab, theta, positions):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": layers, "hidden_size": width,
            "num_attention_heads": heads, "num_key_value_heads": kv_heads, "intermediate_size": ff, "vocab_size": vocab,
            "rope_theta": theta, "rms_norm_eps": 1e-5, "max_position_embeddings": positions, "tie_word_embeddings": False,
            "hidden_act": "silu", "attention_bias": False, "rope_scaling": None, "eos_token_id": 2}


def lufazen(layers, width, ff, heads):
    out = []
    for i in range(layers):
        if i % 4 == 3:
            mixer = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 768, "kv_rank": 512, "scale": 192 ** -0.5,
                     "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 40.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
            if (i // 4) % 2 == 1:
                mixer["kv_from"] = 3
            kind = "latent_attention"
        else:
            mixer = {"heads": heads, "kv_heads": heads, "dim": 128, "vdim": 128, "conv": 4, "decay_rank": 64, "gate_rank": 64}
            kind = "channel_delta"
        out.append({"type": kind, "mixer": mixer, "mlp": {"kind": "dense", "ff": ff, "limit": 7.0}})
    return {"architecture": "Lufazen", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "logit_softcap": 30.0,
            "layers": out, "max_position": 8192}


def fofapel(layers, width, ff, heads):
    out = []
    for i in range(layers):
        mlp = {"kind": "dense", "ff": ff} if i % 4 == 0 else \
            {"kind": "moe", "router": {"experts": 8, "top": 2}, "expert": {"ff": ff // 4, "limit": 7.0},
             "shared": {"ff": ff // 4, "limit": 7.0}}
        out.append({"type": "parallel", "mlp": mlp, "mixer": {
            "left": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "mask": {"size": 512},
                     "rot": {"base": 10000.0, "dims": 128}, "scale": 128 ** -0.5},
            "right": {"heads": width // 64, "dim": 64, "decay_rank": 64}, "left_scale": 1.0, "right_scale": 1.0}})
    return {"architecture": "Fofapel", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "postln_alpha": 2.0,
            "layers": out, "max_position": 8192}


def gesutar(layers, width, ff, heads):
    layer = {"type": "latent_attention",
             "mixer": {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "mask": {"size": 512},
                       "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5},
             "mlp": {"kind": "moe", "router": {"experts": 16, "top": 4, "scale": 1.0, "groups": {"count": 4, "keep": 2}},
                     "expert": {"ff": ff // 8}, "shared": {"ff": ff // 4}}}
    return {"architecture": "Gesutar", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5},
            "embedding": {"scale": 1.0, "bigram": {"buckets": 65521, "mul_prev": 31, "mul_cur": 17}},
            "layers": [layer] * layers, "max_position": 8192}


def vevapel(runs, width, ff, heads):
    mlp = {"kind": "moe", "router": {"experts": 16, "top": 4}, "expert": {"ff": ff // 8}}
    kinds = [{"type": "attention", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128,
                                                         "scale": 128 ** -0.5, "q_temp": {"coef": 0.1, "every": 256}}},
             {"type": "delta", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": heads, "dim": 128, "vdim": 128, "conv": 4}},
             {"type": "attention_2", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128,
                                                           "scale": 128 ** -0.5, "diff": 0.2, "mask": {"size": 512},
                                                           "rot": {"base": 10000.0, "dims": 64}}}]
    return {"architecture": "Vevapel", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 0.5,
            "embedding": {"scale": 1.0}, "layers": [kinds[i % 3] for i in range(runs - 2)],
            "loop": {"start": 1, "stop": 3, "times": 2}, "max_position": 8192}


def mogutar(layers, width, ff, heads):
    mlp = {"kind": "moe", "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}}, "expert": {"ff": ff // 8}}
    both = {"type": "parallel", "mlp": mlp, "mixer": {
        "left": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "conv": 4, "mask": {"size": 512, "keep_first": 4},
                 "scale": 128 ** -0.5, "softcap": 30.0,
                 "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "original": 2048, "fast": 32.0, "slow": 1.0}}},
        "right": {"heads": width // 64, "groups": 2, "state": 128, "vdim": 64, "conv": 4, "norm_groups": 2},
        "left_scale": 1.0, "right_scale": 1.0}}
    linear = {"type": "lightning", "mlp": mlp,
              "mixer": {"heads": heads, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** -(2 + 6.0 * h / heads) for h in range(heads)]}}
    return {"architecture": "Mogutar", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "token_side": {"dim": 64},
            "layers": [linear if i % 2 else both for i in range(layers)], "max_position": 8192}


def nililix(runs, width, ff, heads):
    moe = {"kind": "moe", "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}}, "expert": {"ff": ff // 8}}
    mixer = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "conv": 4, "mask": {"size": 512}, "scale": 128 ** -0.5,
             "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 2048}}}
    return {"architecture": "Nililix", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 0.5,
            "logit_softcap": 30.0, "layers": [{"type": "attention", "mixer": mixer, "mlp": moe if i % 2 else {"kind": "dense", "ff": ff}}
                                              for i in range(runs - 2)],
            "loop": {"start": 1, "stop": 3, "times": 2}, "max_position": 8192}


# The Llama shapes and the designs' sizes of the repository's benchmark.
MODELS = {
    "tinyllama": llama(22, 2048, 32, 4, 5632, 32000, 10000.0, 2048),
    "llama3_8b": llama(32, 4096, 32, 8, 14336, 128256, 500000.0, 8192),
    "lufazen": lufazen(8, 2048, 5632, 16), "fofapel": fofapel(8, 2048, 5632, 16), "gesutar": gesutar(8, 2048, 5632, 16),
    "vevapel": vevapel(8, 2048, 5632, 16), "mogutar": mogutar(8, 2048, 5632, 16), "nililix": nililix(8, 2048, 5632, 16),
}


def is_llama(cfg):
    return "architectures" in cfg


def vocab_of(cfg):
    return cfg["vocab_size"] if is_llama(cfg) else cfg["vocab"]


def order_of(cfg):
    """The layers in the order they run: (layer, pass this run opens or None)."""
    n = cfg["num_hidden_layers"] if is_llama(cfg) else len(cfg["layers"])
    loop = cfg.get("loop")
    if not loop:
        return [(i, None) for i in range(n)]
    return [(i, None) for i in range(loop["start"])] \
        + [(i, t if i == loop["start"] else None) for t in range(loop["times"]) for i in range(loop["start"], loop["stop"])] \
        + [(i, None) for i in range(loop["stop"], n)]


# ------------------------------------------------------------------------------------------------ their tensors
def matrix(out, inner, gain=1.0):
    return ("matrix", (out, inner), gain / math.sqrt(inner))


def vector(n, mean=0.0, std=0.1):
    return ("vector", n if isinstance(n, tuple) else (n,), mean, std)


def taps(channels, n):
    return vector((channels, n), 0.25, 0.25)


def branch(cfg):
    """How far a sublayer's output moves the stream, whose embedding part has unit size: in all about as far again."""
    return 1.0 / math.sqrt(2 * len(order_of(cfg)))


def tensors(cfg):
    """Every tensor of a model by its checkpoint name: (kind, shape, and what `tensor` makes the kind from)."""
    t, b = OrderedDict(), branch(cfg)
    if is_llama(cfg):
        W, F, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
        D = W // cfg["num_attention_heads"]
        Q, K = cfg["num_attention_heads"] * D, cfg["num_key_value_heads"] * D
        t["model.embed_tokens.weight"] = ("matrix", (V, W), 1.0)
        for i in range(cfg["num_hidden_layers"]):
            p = "model.layers.%d." % i
            t.update({p + "input_layernorm.weight": vector(W, 1.0), p + "post_attention_layernorm.weight": vector(W, 1.0),
                      p + "self_attn.q_proj.weight": matrix(Q, W, 1.5), p + "self_attn.k_proj.weight": matrix(K, W, 1.5),
                      p + "self_attn.v_proj.weight": matrix(K, W), p + "self_attn.o_proj.weight": matrix(W, Q, 3 * b),
                      p + "mlp.gate_proj.weight": matrix(F, W), p + "mlp.up_proj.weight": matrix(F, W),
                      p + "mlp.down_proj.weight": matrix(W, F, 2 * b)})
        t["model.norm.weight"] = vector(W, 1.0)
        t["lm_head.weight"] = ("head", (V, W), "model.embed_tokens.weight")
        return t
    W, V, arch = cfg["width"], cfg["vocab"], cfg["architecture"]
    t["embed"] = ("matrix", (V, W), 1.0) if arch in ("Lufazen", "Fofapel") else ("marked", (V, W))
    if arch == "Gesutar":
        t["bigram"] = ("matrix", (cfg["embedding"]["bigram"]["buckets"] + 1, W), 0.3)
    if arch == "Mogutar":
        t["side.embed"] = ("matrix", (V, cfg["token_side"]["dim"] * len(cfg["layers"])), 1.0)
    if arch == "Vevapel":
        t["loop.in"] = ("join", (W, 2 * W), 0.1)
    if cfg.get("loop"):
        t["loop.step"] = vector((cfg["loop"]["times"], W))
    for i, layer in enumerate(cfg["layers"]):
        p = "l%d." % i
        m, mlp = layer["mixer"], layer["mlp"]
        # where norms finish a branch its weight says how far the stream moves; else the branch's last matrix does
        last = {"Lufazen": 1.0, "Fofapel": 0.7, "Gesutar": 2 * b}.get(arch, 1.0)
        if arch == "Lufazen":
            t.update({p + "norm1": vector(W), p + "norm2": vector(W), p + "ls1": vector(W, b, b / 8), p + "ls2": vector(W, b, b / 8)})
        elif arch == "Fofapel":
            t.update({p + "norm1": vector(W, 1.0), p + "norm1.b": vector(W, 0.0, 0.02), p + "norm2": vector(W, 1.0),
                      p + "norm2.b": vector(W, 0.0, 0.02)})
        elif arch == "Gesutar":
            t.update({p + "norm1": vector(W, 1.0), p + "norm2": vector(W, 1.0)})
        elif arch == "Mogutar":
            t.update({p + "norm1": vector(W, b, b / 8), p + "norm2": vector(W, b, b / 8), p + "side.norm": vector(W, b, b / 8)})
        else:
            for n, mean in (("norm1", 1.0), ("norm2", 1.0), ("norm1b", 2 * b), ("norm2b", 2 * b)):
                t[p + n] = vector(W, mean, mean / 8)
                if arch == "Vevapel":
                    t[p + n + ".b"] = vector(W, 0.0, 0.02)
        add = lambda pre, d: t.update({pre + k: v for k, v in d.items()})  # noqa: E731
        kind = layer["type"]
        if kind == "latent_attention":
            H, D, R, VD, C = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            if m.get("q_rank"):
                add(p + "mix.", {"dq": matrix(m["q_rank"], W), "dq.norm": vector(m["q_rank"], 1.0), "uq": matrix(H * (D + R), m["q_rank"], 1.5)})
            else:
                add(p + "mix.", {"q": matrix(H * (D + R), W, 1.5), "sink": vector(H, 0.0, 1.0)})
            if m.get("kv_from") is None:
                add(p + "mix.", {"dkv": matrix(C + R, W), "dkv.norm": vector(C, 1.0)})
            add(p + "mix.", {"uk": matrix(H * D, C, 1.5), "uv": matrix(H * VD, C),
                             "g": matrix(H if arch == "Lufazen" else H * VD, W), "o": matrix(W, H * VD, last)})
        elif kind in ("channel_delta", "delta"):
            H, D, VD, n = m["heads"], m["dim"], m["vdim"], m["conv"]
            for x, c in (("q", m["kv_heads"] * D), ("k", m["kv_heads"] * D), ("v", H * VD)):
                add(p + "mix.", {x: matrix(c, W), x + ".conv": taps(c, n)})
            add(p + "mix.", {"b": matrix(H, W), "A_log": vector(H, 0.0, 0.5), "norm": vector(VD, 1.0), "o": matrix(W, H * VD, last)})
            if kind == "delta":
                add(p + "mix.", {"a": matrix(H, W), "dt_bias": vector(H, -3.0, 1.0), "g": matrix(H * VD, W)})
            else:
                r, s = m["decay_rank"], m["gate_rank"]
                add(p + "mix.", {"a1": matrix(r, W), "a2": matrix(H * D, r), "dt_bias": vector(H * D, -3.0, 1.0),
                                 "g1": matrix(s, W), "g2": matrix(H * VD, s)})
        elif kind == "parallel" and arch == "Fofapel":
            l, r = m["left"], m["right"]
            H, G, D = l["heads"], l["kv_heads"], l["dim"]
            # the queries and keys of these heads have unit root mean square, so their scores need no gain
            add(p + "mix.left.", {"q": matrix(H * D, W), "k": matrix(G * D, W), "q.b": vector(H * D), "k.b": vector(G * D),
                                  "g": matrix(H, W), "o": matrix(W, H * D, last)})
            n = r["heads"] * r["dim"]
            add(p + "mix.right.", {"mu." + x: vector(W, 0.5, 0.2) for x in "rkvgw"})
            add(p + "mix.right.", {x: matrix(n, W) for x in "rkvg"})
            add(p + "mix.right.", {"w1": matrix(r["decay_rank"], W), "w2": matrix(n, r["decay_rank"], 0.5), "w0": vector(n, -2.0, 1.0),
                                   "u": vector((r["heads"], r["dim"]), 0.5, 0.3), "norm": vector(n, 1.0), "o": matrix(W, n, last)})
        else:
            l, pre = (m["left"], p + "mix.left.") if kind == "parallel" else (m, p + "mix.")
            H, G, D, VD = l["heads"], l.get("kv_heads", l["heads"]), l["dim"], l["vdim"]
            if kind == "lightning":
                add(pre, {x: matrix(H * D, W) for x in "qk"})
                add(pre, {"v": matrix(H * VD, W), "g": matrix(H * VD, W), "norm": vector(H * VD, 1.0), "o": matrix(W, H * VD)})
            else:
                maps = 2 if kind == "attention_2" else 1
                add(pre, {"q": matrix(H * maps * D, W, 1.5), "k": matrix(G * maps * D, W, 1.5), "v": matrix(G * VD, W), "o": matrix(W, H * VD)})
                if arch != "Nililix":
                    add(pre, {"q.b": vector(H * maps * D), "k.b": vector(G * maps * D), "v.b": vector(G * VD)})
                if l.get("conv"):
                    add(pre, {"q.conv": taps(H * D, l["conv"]), "k.conv": taps(G * D, l["conv"]), "v.conv": taps(G * VD, l["conv"])})
                if arch == "Nililix":
                    add(pre, {"sink": vector(H, 0.0, 1.0), "g": matrix(H, W)})
                elif arch == "Mogutar":
                    add(pre, {"q.norm": vector(D, 1.2), "k.norm": vector(D, 1.2)})
                elif kind == "attention":
                    add(pre, {"q.norm": vector(H * D, 1.2), "k.norm": vector(G * D, 1.2), "g": matrix(H, W), "o.b": vector(W, 0.0, 0.02)})
                else:
                    add(pre, {"g": matrix(H * VD, W)})
                    add(pre, {x: vector(D) for x in ("lq1", "lk1", "lq2", "lk2")})
            if kind == "parallel":
                r = m["right"]
                h, vd, inner = r["heads"], r["vdim"], r["heads"] * r["vdim"]
                c = inner + 2 * r["groups"] * r["state"]
                add(p + "mix.right.", {"in": matrix(inner + c + h, W), "conv": taps(c, r["conv"]), "conv.b": vector(c),
                                       "dt_bias": vector(h, -3.0, 1.0), "A_log": vector(h, 0.5, 0.5), "D": vector(h, 1.0),
                                       "norm": vector(inner, 1.0), "o": matrix(W, inner)})
        pre = p + "mlp."
        if mlp["kind"] == "dense":
            if arch != "Nililix":
                add(pre, {"gate": matrix(mlp["ff"], W)})
            add(pre, {"up": matrix(mlp["ff"], W), "down": matrix(W, mlp["ff"], last)})
        else:
            r, f = mlp["router"], mlp["expert"]["ff"]
            gated = arch != "Gesutar"
            names = ["e%d." % e for e in range(r["experts"])] + (["shared."] if mlp.get("shared") else [])
            for n in names:
                f = (mlp["shared"] if n == "shared." else mlp["expert"])["ff"]
                if gated:
                    add(pre + n, {"gate": matrix(f, W)})
                add(pre + n, {"up": matrix(f, W), "down": matrix(W, f, last)})
            if arch == "Fofapel":
                add(pre, {"table": ("table", (V, r["top"]), r["experts"]), "shared.sg": matrix(1, W)})
            else:
                add(pre, {"router": ("router", (r["experts"], W), i)})
                if arch == "Vevapel":
                    add(pre, {"router.b": vector(r["experts"])})
                elif arch != "Gesutar":
                    add(pre, {"correction": vector(r["experts"], 0.0, 0.02)})
        if arch == "Mogutar":
            add(p + "side.", {"gate": matrix(cfg["token_side"]["dim"], W), "proj": matrix(W, cfg["token_side"]["dim"])})
    t["final.norm"] = vector(W, 0.0 if arch == "Lufazen" else 1.0)
    if arch in ("Fofapel", "Vevapel"):
        t["final.norm.b"] = vector(W, 0.0, 0.02)
    if arch != "Vevapel":                                  # Vevapel's head is its embedding
        t["head"] = ("head", (V, W), "embed")
    return t


def successor(cfg):
    """The likeliest token behind every token: the head's row of it is the token's embedding."""
    V = vocab_of(cfg)
    if cfg.get("architecture") == "Vevapel":
        return torch.arange(V, device=DEVICE)
    return torch.randperm(V, generator=torch.Generator(device=DEVICE).manual_seed(7), device=DEVICE)


def tensor(cfg, name, what, elt):
    """One tensor, on the device: matrices in `elt` (the engine's type), vectors in float32."""
    g = torch.Generator(device=DEVICE).manual_seed(zlib.crc32(name.encode()))
    if what[0] == "head":
        # the likeliest token's logit lies near 20 where the others' have a standard deviation near 1
        source = tensor(cfg, what[2], tensors(cfg)[what[2]], elt).float()
        to = successor(cfg)
        out = torch.empty_like(source)
        out[to] = source / math.sqrt(source.shape[1])
        return out.to(elt)
    if what[0] == "table":
        start = torch.randint(0, what[2], (what[1][0], 1), generator=g, device=DEVICE)
        return ((start + torch.arange(what[1][1], device=DEVICE)) % what[2]).to(torch.int32)
    z = torch.randn(what[1], generator=g, device=DEVICE)
    if what[0] == "marked":
        # the first 16 numbers say which experts suit a token, as plainly as trained routers see it: two of four groups,
        # two experts in each, so that a choice does not hang on a rounding error
        group = torch.rand(z.shape[0], 4, generator=g, device=DEVICE).argsort(dim=1)[:, :2, None]
        member = torch.rand(z.shape[0], 2, 4, generator=g, device=DEVICE).argsort(dim=2)[:, :, :2]
        z[:, :16] = 0.3 * z[:, :16].scatter(1, (4 * group + member).flatten(1), 27.0)
        return z.to(elt)
    if what[0] == "router":                                # every layer reads the marks from another group on
        z = z * (0.3 / math.sqrt(what[1][1]))
        e = torch.arange(what[1][0], device=DEVICE)
        z[e, (e + 4 * what[2]) % 16] = 0.4
        return z.to(elt)
    if what[0] == "join":                                  # [the stream | the embedding]: mostly the first passes on
        return (z * (what[2] / math.sqrt(what[1][1])) + torch.eye(what[1][0], device=DEVICE).repeat(1, 2) * 0.5).to(elt)
    return (z * what[2]).to(elt) if what[0] == "matrix" else z * what[3] + what[2]


# --------------------------------------------------------------------------------------------------- the cases
def case(name, model, dtype="bfloat16", prompts=1, shortest=1, longest=1, new=0, budget=4096, sample=False):
    c = {"model": model, "dtype": dtype, "prompts": prompts, "shortest": shortest, "longest": longest, "new": new,
         "budget": budget, "sample": sample}
    return dict({"name": name}, **c) if name else c


def listed():
    return [
        # a question and the first words of an answer: every launch counts, nothing fills the chip
        case("tinyllama_short", "tinyllama", prompts=1, shortest=9, longest=9, new=8),
        # the headline: eight requests decoding behind prompts of 512 tokens
        case("tinyllama_batch8", "tinyllama", prompts=8, shortest=512, longest=512, new=64),
        # a full server of short chats, drawn from the distribution the reference draws from by default
        case("tinyllama_batch64", "tinyllama", prompts=64, shortest=13, longest=131, new=32, sample=True),
        # one prompt as long as the model's context allows: the time to its first token
        case("tinyllama_prompt2047", "tinyllama", prompts=1, shortest=2047, longest=2047),
        # the true 32-bit path: ragged prompts and their answers
        case("tinyllama_float32", "tinyllama", "float32", prompts=8, shortest=17, longest=203, new=16),
        # a larger model under load: prompts of 130 to 4,100 tokens in portions of 2,048 beside decoded tokens
        case("llama3_8b_mixed", "llama3_8b", prompts=8, shortest=130, longest=4099, new=16, budget=2048),
        # the other designs, each with a batch of ragged prompts and their answers
        case("lufazen_batch6", "lufazen", prompts=6, shortest=67, longest=801, new=16),
        case("fofapel_batch6", "fofapel", prompts=6, shortest=67, longest=801, new=16),
        case("gesutar_batch6", "gesutar", prompts=6, shortest=67, longest=801, new=16),
        case("vevapel_batch6", "vevapel", prompts=6, shortest=67, longest=801, new=16),
        case("mogutar_batch6", "mogutar", prompts=6, shortest=67, longest=801, new=16),
        case("nililix_batch6", "nililix", prompts=6, shortest=67, longest=801, new=16),
    ]


def draw(rng: random.Random):
    """Batches of 1 to 64 requests with prompts of 2 to 4,000 tokens and up to 64 new ones, on any of the models."""
    log = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    while True:
        model = rng.choice(["tinyllama"] * 6 + ["llama3_8b"] + [m for m in MODELS if m not in ("tinyllama", "llama3_8b")])
        dtype = "float32" if model == "tinyllama" and rng.random() < 0.25 else "bfloat16"
        prompts = log(1, 64)
        a, b = sorted(log(2, 1900 if model == "tinyllama" else 4000) for _ in range(2))
        c = case(None, model, dtype, prompts, a, b if prompts > 1 else a, log(1, 65) - 1, rng.choice([512, 1024, 2048, 4096]),
                 rng.random() < 0.3)
        total, most = sum(lengths(c)), {"llama3_8b": 9000, "tinyllama": 16000 if dtype == "bfloat16" else 2500}.get(model, 8000)
        if total <= most and (model != "llama3_8b" or c["new"] <= 16):
            return c


def lengths(c):
    """The prompts' lengths: from the shortest to the longest in equal ratios, the long ones spread among the short."""
    n, a, b = c["prompts"], c["shortest"], c["longest"]
    got = [int(round(a * (b / a) ** (i / max(1, n - 1)))) for i in range(n)]
    stride = next(s for s in (5, 7, 11, 13, 1) if math.gcd(s, n) == 1)
    return [got[i * stride % n] for i in range(n)]


def schedule(c):
    """The engine's order of work: decoded tokens first, then prompts in the order they came, `budget` tokens a step.
    Returns (rows of every step, the step at which each request's last prompt token is computed)."""
    left, first, steps = lengths(c), [None] * c["prompts"], []
    while None in first or len(steps) <= max(first) + c["new"]:
        s = len(steps)
        rows = sum(1 for f in first if f is not None and f < s <= f + c["new"])
        room = c["budget"] - rows
        for i, n in enumerate(left):
            take = min(n, room)
            if take:
                left[i] -= take
                room -= take
                rows += take
                if not left[i]:
                    first[i] = s
        steps.append(rows)
    return steps, first


_engines: "OrderedDict[tuple, object]" = OrderedDict()


def engine_of(c):
    """The live engine of a case's model (one is kept: what a serving program has)."""
    key = (c["model"], c["dtype"], c["budget"])
    if key not in _engines:
        _engines.clear()
        torch.cuda.empty_cache()
        cfg = MODELS[c["model"]]
        engine = Engine(config=cfg, dtype=c["dtype"], max_num_seqs=64, max_num_batched_tokens=c["budget"], max_cache_tokens=24576)
        weights = Checkpoint()
        elt = getattr(torch, c["dtype"])
        for name, what in tensors(cfg).items():
            weights.set_tensor(name, tensor(cfg, name, what, elt))
        load_weights(engine.decoder, weights)
        _engines[key] = (engine, set())
    return _engines[key]


def prompts_of(c, seed):
    g = torch.Generator().manual_seed(int(seed))
    return [torch.randint(0, vocab_of(MODELS[c["model"]]), (n,), generator=g).tolist() for n in lengths(c)]


def prepare(c, seed):
    engine, warm = engine_of(c)
    params = SamplingParams(max_new_tokens=c["new"] + 1, do_sample=c["sample"], seed=int(seed), ignore_eos=True)
    state = {"engine": engine, "prompts": prompts_of(c, seed), "params": params, "new": c["new"]}
    shape = repr(sorted((k, v) for k, v in c.items() if k != "name"))
    if shape not in warm:                                  # a server meets its shapes of step before its users do
        for k in range(3):
            run(dict(state, prompts=prompts_of(c, 1000 + k)))
        warm.add(shape)
    return state


def run(state):
    """Requests that are done early leave the batch; the logits are those of the requests that are done last."""
    engine, params, new = state["engine"], state["params"], state["new"]
    ids = [engine.add_request(p, params) for p in state["prompts"]]
    requests = [engine.requests[i] for i in ids]
    while (left := max(max(1, new) - len(r.output) for r in requests)) > 0:
        engine.step(max_decode_steps=left)
    if new:
        live = [r for r in requests if r.status != "finished"]
        logits = engine.runner.step([StepEntry(r.req_id, r.output[-1:], [0]) for r in live], use_graph=True)
        for r in live:
            engine.abort(r.req_id)
    else:
        logits = engine.runner.last_logits.clone()
    tokens = torch.tensor([engine.release(i).output[:max(1, new)] for i in ids])
    return {"tokens": tokens, "logits": logits}


# ------------------------------------------------------------------------------------------------------ figures
def work(c):
    """Weights once a step (no step can begin before the one ahead of it is done, and no model here fits a cache; of the
    experts those that a step's rows can reach), the cached keys and values, the logits; two operations a weight and
    row, the scores and the sums over values."""
    cfg = MODELS[c["model"]]
    steps, _ = schedule(c)
    size = 2 if c["dtype"] == "bfloat16" else 4
    runs = {}
    for i, _ in order_of(cfg):
        runs[i] = runs.get(i, 0) + 1
    byte_s, flops = 0.0, 0.0
    rows_total, outs = sum(steps), c["prompts"] * (c["new"] + 1)
    for name, what in tensors(cfg).items():
        n = math.prod(what[1])
        if name in ("embed", "side.embed", "bigram", "model.embed_tokens.weight"):
            byte_s += size * rows_total * what[1][1]
            if name == "embed" and cfg.get("architecture") == "Vevapel":
                byte_s, flops = byte_s + size * n * len(steps), flops + 2.0 * n * outs
            continue
        if what[0] == "table":
            byte_s += 4.0 * rows_total * what[1][1]
            continue
        part = name.split(".")
        times, share, reached = 1, 1.0, len(steps)
        if part[0][0] == "l" and part[0][1:].isdigit():
            i = int(part[0][1:])
            times = runs[i]
            if len(part) > 2 and part[1] == "mlp" and part[2][0] == "e" and part[2][1:].isdigit():
                r = cfg["layers"][i]["mlp"]["router"]
                share = r["top"] / r["experts"]
                reached = sum(1 - (1 - share) ** rows for rows in steps)
        byte_s += (size if what[0] != "vector" else 4) * n * times * reached
        if what[0] in ("matrix", "join", "router"):
            flops += 2.0 * n * times * rows_total * share
        elif what[0] == "head":
            flops += 2.0 * n * outs
    byte_s += 4.0 * vocab_of(cfg) * c["prompts"] + 8.0 * outs
    ends = [n + c["new"] for n in lengths(c)]
    for i, _ in order_of(cfg):
        layer = cfg["layers"][i] if not is_llama(cfg) else None
        m = layer["mixer"] if layer else {"heads": cfg["num_attention_heads"], "kv_heads": cfg["num_key_value_heads"],
                                          "dim": cfg["hidden_size"] // cfg["num_attention_heads"]}
        for part in ([m["left"], m["right"]] if "left" in m else [m]):
            H, D = part["heads"], part.get("dim", part.get("state"))
            VD = part.get("vdim", D)
            attends = not layer or "attention" in layer["type"] or part is m.get("left")
            for n, end in zip(lengths(c), ends):
                if not attends:                            # a recurrence: the state decays, takes a product, gives one
                    flops += 6.0 * end * H * D * VD
                    byte_s += 8.0 * H * D * VD * (c["new"] + 1)
                    continue
                window = (part.get("mask") or {}).get("size") or end
                maps = 2 if layer and layer["type"] == "attention_2" else 1
                rot = part.get("rot_dim", 0)
                seen = sum(min(p + 1, window) for p in range(end))
                flops += 2.0 * H * seen * (maps * (D + rot + VD))
                a_key = part["kv_rank"] + rot if rot else part.get("kv_heads", H) * (maps * D + VD)
                byte_s += size * a_key * (end + sum(min(p + 1, window) for p in range(n, end)))
    return {"bytes": byte_s, "flops": flops}


def tolerance(c):
    return {"rel": 1e-5, "max": 1e-4} if c["dtype"] == "float32" else {"rel": 2e-2, "max": 0.15}


# ------------------------------------------------------------------------------- the same in 64 bits, plain torch
def unit(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def layer_norm(x, w, b, eps):
    d = x - x.mean(dim=-1, keepdim=True)
    return unit(d, eps) * w + b


def silu(z):
    return z * torch.sigmoid(z)


def gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def softplus(z):
    return torch.nn.functional.softplus(z, threshold=700.0)


def swish(g, u, limit):
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


def frequencies(rot):
    """One frequency per rotated pair and what multiplies cosine and sine."""
    n, base, s = rot["dims"] // 2, rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / rot["dims"]) for i in range(n)]
    if not s:
        return f, 1.0
    if "fast" in s:                                        # YaRN: slow pairs are stretched
        index = lambda turns: rot["dims"] * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(index(s["fast"])), 0), min(math.ceil(index(s["slow"])), rot["dims"] - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(n)]
        return [a / s["factor"] * r + a * (1 - r) for a, r in zip(f, ramp)], 0.1 * math.log(s["factor"]) + 1.0
    out = []
    for a in f:                                            # Llama 3.1: long waves are stretched, those between in part
        wave = 2 * math.pi / a
        keep = min(max((s["original"] / wave - s["low"]) / (s["high"] - s["low"]), 0.0), 1.0)
        out.append((1 - keep) * a / s["factor"] + keep * a)
    return out, 1.0


def rotate(x, positions, rot, pairs=False):
    """x [T, ..., D]: the first rot["dims"] numbers turn, i with i + dims/2, or 2i with 2i + 1."""
    dims = rot["dims"]
    f, mag = frequencies(rot)
    a = positions.double()[:, None] * torch.tensor(f, dtype=torch.float64, device=x.device)
    a = a.reshape([x.shape[0]] + [1] * (x.dim() - 2) + [dims // 2])
    cos, sin = torch.cos(a) * mag, torch.sin(a) * mag
    out = x.clone()
    one, two = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    u, v = x[..., one], x[..., two]
    out[..., one], out[..., two] = u * cos - v * sin, v * cos + u * sin
    return out


class Plain:
    """A model's forward pass over several whole sequences, end to end in one list of rows."""

    def __init__(self, cfg, elt, sequences):
        self.cfg, self.elt, self.all = cfg, elt, tensors(cfg)
        self.sizes = [len(s) for s in sequences]
        self.tokens = torch.tensor([t for s in sequences for t in s], device=DEVICE)
        self.positions = torch.cat([torch.arange(n, device=DEVICE) for n in self.sizes])
        self.kept = {}

    def w(self, name):
        return tensor(self.cfg, name, self.all[name], self.elt).double()

    def rows(self, x):
        return torch.split(x, self.sizes)

    def padded(self, x):
        return torch.nn.utils.rnn.pad_sequence(self.rows(x), batch_first=True)

    def flat(self, x):
        return torch.cat([x[r, :n] for r, n in enumerate(self.sizes)])

    def before(self, x, back=1):
        """The row `back` places ahead of each in its sequence (zeros ahead of the first)."""
        out = torch.zeros_like(x)
        out[back:] = x[:-back] if back < x.shape[0] else 0.0
        return torch.where((self.positions >= back).reshape([-1] + [1] * (x.dim() - 1)), out, torch.zeros_like(x))

    def conv(self, x, w):
        n = w.shape[1]
        return sum((self.before(x, n - 1 - j) if j < n - 1 else x) * w[:, j] for j in range(n))

    def attend(self, q, k, v, scale, window=0, first=0, chunk=0, cap=None, sink=None):
        """q [N, H, D], k [N, G, D], v [N, G, V]; `sink` [H]: one more score without a value."""
        H, G = q.shape[1], k.shape[1]
        out = []
        for qs, ks, vs in zip(self.rows(q), self.rows(k), self.rows(v)):
            T = qs.shape[0]
            i = torch.arange(T, device=DEVICE)
            back = i[:, None] - i[None, :]
            seen = back >= 0
            if window:
                seen &= (back < window) | (i[None, :] < first)
            if chunk:
                seen &= (i[:, None] // chunk) == (i[None, :] // chunk)
            got = torch.empty(T, H, v.shape[-1], dtype=q.dtype, device=DEVICE)
            for h in range(H):
                g = h // (H // G)
                s = (qs[:, h] @ ks[:, g].T) * scale
                if cap:
                    s = cap * torch.tanh(s / cap)
                s = s.masked_fill_(~seen, float("-inf"))
                if sink is not None:
                    s = torch.cat([s, sink[h].expand(T, 1)], dim=1)
                got[:, h] = torch.softmax(s, dim=-1)[:, :T] @ vs[:, g]
            out.append(got)
        return torch.cat(out)

    def scan(self, step, state, *xs):
        """`step(state, rows of token t) -> (state, result)` over all sequences at once."""
        xs = [self.padded(x) for x in xs]
        out = []
        for t in range(max(self.sizes)):
            state, o = step(state, *(x[:, t] for x in xs))
            out.append(o)
        return self.flat(torch.stack(out, dim=1))

    # ------------------------------------------------------------------------------------------------- mixers
    def zeros(self, *shape):
        return torch.zeros(len(self.sizes), *shape, dtype=torch.float64, device=DEVICE)

    def latent_attention(self, h, p, m, i):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        H, D, C = m["heads"], m["dim"], m["kv_rank"]
        pairs = not m.get("q_rank")
        if pairs:
            q = h @ w("q").T
        else:
            q = (unit(h @ w("dq").T, eps) * w("dq.norm")) @ w("uq").T
        q = q.reshape(N, H, -1)
        if m.get("kv_from") is None:
            d = h @ w("dkv").T
            self.kept[i] = unit(d[:, :C], eps) * w("dkv.norm"), rotate(d[:, C:], self.positions, m["rot"], pairs)
        c, kr = self.kept[i if m.get("kv_from") is None else m["kv_from"]]
        q = torch.cat([q[..., :D], rotate(q[..., D:], self.positions, m["rot"], pairs)], dim=-1)
        k = torch.cat([(c @ w("uk").T).reshape(N, H, D), kr[:, None, :].expand(N, H, kr.shape[1])], dim=-1)
        v = (c @ w("uv").T).reshape(N, H, -1)
        o = self.attend(q, k, v, m["scale"], (m.get("mask") or {}).get("size", 0), sink=w("sink") if pairs else None)
        g = torch.sigmoid(h @ w("g").T)
        return (o * g[:, :, None] if not pairs else o * g.reshape(o.shape)).reshape(N, -1) @ w("o").T

    def any_delta(self, h, p, m, by_channel):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (silu(self.conv(h @ w(n).T, w(n + ".conv"))) for n in "qkv")
        length = lambda x: x / torch.sqrt((x * x).sum(dim=-1, keepdim=True) + 1e-6)  # noqa: E731
        q = (length(q.reshape(N, G, D)) * D ** -0.5).repeat_interleave(H // G, dim=1)
        k = length(k.reshape(N, G, D)).repeat_interleave(H // G, dim=1)
        a = h @ w("a1").T @ w("a2").T if by_channel else h @ w("a").T
        rate = torch.exp(w("A_log"))[None, :, None]
        decay = torch.exp(-rate * softplus(a + w("dt_bias")).reshape(N, H, -1))

        def step(S, q, k, v, beta, decay):
            S = S * decay[..., None]
            u = beta[..., None] * (v - (S * k[..., None]).sum(dim=-2))
            S = S + k[..., None] * u[..., None, :]
            return S, (S * q[..., None]).sum(dim=-2)

        o = self.scan(step, self.zeros(H, D, V), q, k, v.reshape(N, H, V), torch.sigmoid(h @ w("b").T), decay)
        o = (unit(o, eps) * w("norm")).reshape(N, -1)
        g = torch.sigmoid(h @ w("g1").T @ w("g2").T) if by_channel else silu(h @ w("g").T)
        return (o * g) @ w("o").T

    def channel_delta(self, h, p, m, i):
        return self.any_delta(h, p, m, True)

    def delta(self, h, p, m, i):
        return self.any_delta(h, p, m, False)

    def window_attention(self, h, p, m):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        q = (h @ w("q").T + w("q.b")).reshape(N, m["heads"], -1)
        v = (h @ w("k").T + w("k.b")).reshape(N, m["kv_heads"], -1)
        q, k = (unit(rotate(x, self.positions, m["rot"], True), eps) for x in (q, v))
        o = self.attend(q, k, v, m["scale"], m["mask"]["size"], sink=torch.zeros(m["heads"], dtype=h.dtype, device=DEVICE))
        return (o * torch.sigmoid(h @ w("g").T)[:, :, None]).reshape(N, -1) @ w("o").T

    def time_mix(self, h, p, m):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        H, D = m["heads"], m["dim"]
        mix = lambda n: h + (self.before(h) - h) * w("mu." + n)  # noqa: E731
        r, k, v = ((mix(n) @ w(n).T).reshape(N, H, D) for n in "rkv")
        decay = torch.exp(-torch.exp(torch.tanh(mix("w") @ w("w1").T) @ w("w2").T + w("w0"))).reshape(N, H, D)
        now = w("u")[None, :, :, None]

        def step(S, r, k, v, decay):
            kv = k[..., None] * v[..., None, :]
            return decay[..., None] * S + kv, ((S + now * kv) * r[..., None]).sum(dim=-2)

        o = unit(self.scan(step, self.zeros(H, D, D), r, k, v, decay), eps).reshape(N, -1) * w("norm")
        return (o * silu(mix("g") @ w("g").T)) @ w("o").T

    def mamba(self, h, p, m):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        H, V, S, G = m["heads"], m["vdim"], m["state"], m["groups"]
        z, x, dt = torch.split(h @ w("in").T, [H * V, H * V + 2 * G * S, H], dim=1)
        x = silu(self.conv(x, w("conv")) + w("conv.b"))
        x, B, C = torch.split(x, [H * V, G * S, G * S], dim=1)
        x = x.reshape(N, H, V)
        B, C = (y.reshape(N, G, S).repeat_interleave(H // G, dim=1) for y in (B, C))
        dt = softplus(dt + w("dt_bias"))
        o = self.decayed(torch.exp(-torch.exp(w("A_log")) * dt), C, B, dt[..., None] * x) + w("D")[:, None] * x
        o = o.reshape(N, -1) * silu(z)
        return (unit(o.reshape(N, m["norm_groups"], -1), eps).reshape(N, -1) * w("norm")) @ w("o").T

    def decayed(self, a, q, k, v):
        def step(S, a, q, k, v):
            S = a[..., None, None] * S + k[..., None] * v[..., None, :]
            return S, (S * q[..., None]).sum(dim=-2)
        return self.scan(step, self.zeros(q.shape[1], q.shape[2], v.shape[2]), a, q, k, v)

    def parallel(self, h, p, m, i):
        if self.cfg["architecture"] == "Fofapel":
            left, right = self.window_attention(h, p + "left.", m["left"]), self.time_mix(h, p + "right.", m["right"])
        else:
            left, right = self.attention(h, p + "left.", m["left"], i), self.mamba(h, p + "right.", m["right"])
        return m["left_scale"] * left + m["right_scale"] * right

    def lightning(self, h, p, m, i):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        q, k, v = (silu(h @ w(n).T).reshape(N, m["heads"], -1) for n in "qkv")
        a = torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE).expand(N, -1)
        o = unit(self.decayed(a, q, k, v).reshape(N, -1), eps) * w("norm")
        return (o * torch.sigmoid(h @ w("g").T)) @ w("o").T

    def attention(self, h, p, m, i):
        arch, w, N, eps = self.cfg["architecture"], lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        q, k, v = (h @ w(n).T for n in "qkv")
        if arch != "Nililix":
            q, k, v = q + w("q.b"), k + w("k.b"), v + w("v.b")
        if m.get("conv"):
            q, k, v = self.conv(q, w("q.conv")), self.conv(k, w("k.conv")), self.conv(v, w("v.conv"))
        if arch == "Vevapel":
            q, k = unit(q, eps) * w("q.norm"), unit(k, eps) * w("k.norm")
            t = m["q_temp"]
            turns = torch.div(self.positions + 1, t["every"], rounding_mode="floor").double()
            q = q * (1.0 + t["coef"] * torch.log(turns + 1.0))[:, None]
        q, k, v = q.reshape(N, m["heads"], -1), k.reshape(N, m["kv_heads"], -1), v.reshape(N, m["kv_heads"], -1)
        if arch == "Mogutar":
            q, k = unit(q, eps) * w("q.norm"), unit(k, eps) * w("k.norm")
        if m.get("rot"):
            q, k = (rotate(x, self.positions, m["rot"], arch == "Nililix") for x in (q, k))
        mask = m.get("mask") or {}
        o = self.attend(q, k, v, m["scale"], mask.get("size", 0), mask.get("keep_first", 0), cap=m.get("softcap"),
                        sink=w("sink") if arch == "Nililix" else None)
        if arch != "Mogutar":
            o = o * torch.sigmoid(h @ w("g").T)[:, :, None]
        o = o.reshape(N, -1) @ w("o").T
        return o + w("o.b") if arch == "Vevapel" else o

    def attention_2(self, h, p, m, i):
        w, N, eps = lambda n: self.w(p + n), h.shape[0], self.cfg["norm"]["eps"]
        H, G = m["heads"], m["kv_heads"]
        q, k = ((h @ w(n).T + w(n + ".b")).reshape(N, x, 2, -1) for n, x in (("q", H), ("k", G)))
        v = (h @ w("v").T + w("v.b")).reshape(N, G, -1)
        q, k = rotate(q, self.positions, m["rot"]), rotate(k, self.positions, m["rot"])
        a, b = (self.attend(q[:, :, j], k[:, :, j], v, m["scale"], chunk=m["mask"]["size"]) for j in (0, 1))
        lam = torch.exp((w("lq1") * w("lk1")).sum()) - torch.exp((w("lq2") * w("lk2")).sum()) + m["diff"]
        o = unit(a - lam * b, eps) * (1.0 - m["diff"])
        return (o.reshape(N, -1) * torch.sigmoid(h @ w("g").T)) @ w("o").T

    # ------------------------------------------------------------------------------------------ feed-forwards
    def unit_ff(self, h, p, limit):
        arch = self.cfg["architecture"]
        u = h @ self.w(p + "up").T
        if p + "gate" not in self.all:
            u = u.clamp(min=0.0) ** 2
        else:
            g = h @ self.w(p + "gate").T
            u = swish(g, u, limit) if limit else gelu(g) * u if arch == "Fofapel" else silu(g) * u
        return u @ self.w(p + "down").T

    def choose(self, h, p, r):
        """(experts, their weights), [N, top] each."""
        arch, E, top = self.cfg["architecture"], r["experts"], r["top"]
        z = h @ self.w(p + "router").T
        if arch == "Vevapel":
            best = (z + self.w(p + "router.b")).topk(top, dim=-1)
            return best.indices, torch.softmax(best.values, dim=-1)
        s = torch.softmax(z, dim=-1) if arch == "Gesutar" else torch.sigmoid(z)
        pick = s if arch == "Gesutar" else s + self.w(p + "correction")
        g = r["groups"]
        groups = pick.reshape(-1, g["count"], E // g["count"])
        rank = groups.max(dim=-1).values if arch == "Gesutar" else groups.topk(2, dim=-1).values.sum(dim=-1)
        kept = torch.zeros_like(rank, dtype=torch.bool).scatter_(1, rank.topk(g["keep"], dim=-1).indices, True)
        idx = pick.masked_fill(~kept.repeat_interleave(E // g["count"], dim=1), float("-inf")).topk(top, dim=-1).indices
        wts = s.gather(1, idx)
        if arch == "Gesutar":
            wts = wts / (wts.sum(dim=-1, keepdim=True) + 1e-20) * r["scale"]
        return idx, wts

    def feed_forward(self, h, p, mlp):
        if mlp["kind"] == "dense":
            return self.unit_ff(h, p, mlp.get("limit"))
        r = mlp["router"]
        if p + "table" in self.all:
            idx = tensor(self.cfg, p + "table", self.all[p + "table"], self.elt)[self.tokens].long()
            wts = torch.full(idx.shape, 1.0 / r["top"], dtype=h.dtype, device=DEVICE)
        else:
            idx, wts = self.choose(h, p, r)
        out = torch.zeros_like(h)
        for e in range(r["experts"]):
            row, k = (idx == e).nonzero(as_tuple=True)
            if row.numel():
                out[row] += wts[row, k][:, None] * self.unit_ff(h[row], p + "e%d." % e, mlp["expert"].get("limit"))
        if mlp.get("shared"):
            y = self.unit_ff(h, p + "shared.", mlp["shared"].get("limit"))
            out += y * torch.sigmoid(h @ self.w(p + "shared.sg").T) if p + "shared.sg" in self.all else y
        return out

    # -------------------------------------------------------------------------------------------------- models
    def logits(self, rows):
        return self.llama(rows) if is_llama(self.cfg) else self.design(rows)

    def table_rows(self, name, ids, cut=slice(None)):
        return tensor(self.cfg, name, self.all[name], self.elt)[ids][:, cut].double()

    def llama(self, rows):
        cfg, eps = self.cfg, self.cfg["rms_norm_eps"]
        H, G = cfg["num_attention_heads"], cfg["num_key_value_heads"]
        D = cfg["hidden_size"] // H
        rot = {"dims": D, "base": cfg["rope_theta"]}
        x = self.table_rows("model.embed_tokens.weight", self.tokens)
        for i in range(cfg["num_hidden_layers"]):
            w = lambda n: self.w("model.layers.%d.%s.weight" % (i, n))  # noqa: E731
            h = unit(x, eps) * w("input_layernorm")
            q, k, v = ((h @ w("self_attn." + n).T).reshape(-1, g, D) for n, g in (("q_proj", H), ("k_proj", G), ("v_proj", G)))
            o = self.attend(rotate(q, self.positions, rot), rotate(k, self.positions, rot), v, D ** -0.5)
            x = x + o.reshape(-1, H * D) @ w("self_attn.o_proj").T
            h = unit(x, eps) * w("post_attention_layernorm")
            x = x + (silu(h @ w("mlp.gate_proj").T) * (h @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
        return (unit(x[rows], eps) * self.w("model.norm.weight")) @ self.w("lm_head.weight").T

    def design(self, rows):
        cfg, arch, eps, w = self.cfg, self.cfg["architecture"], self.cfg["norm"]["eps"], self.w
        x = self.table_rows("embed", self.tokens)
        if arch == "Gesutar":
            b = cfg["embedding"]["bigram"]
            pair = (self.before(self.tokens) * b["mul_prev"] + self.tokens * b["mul_cur"]) % b["buckets"]
            x = x * cfg["embedding"]["scale"] + self.table_rows("bigram", torch.where(self.positions == 0, b["buckets"], pair))
        x0, m = x, cfg.get("residual_mult", 1.0)
        norm = lambda n, y: layer_norm(y, w(n), w(n + ".b"), eps) if n + ".b" in self.all else \
            unit(y, eps) * (w(n) + (1.0 if arch == "Lufazen" else 0.0))  # noqa: E731
        for i, opens in order_of(cfg):
            if opens is not None:
                if arch == "Vevapel":
                    x = torch.cat([x, x0], dim=-1) @ w("loop.in").T
                x = x + w("loop.step")[opens]
            layer, p = cfg["layers"][i], "l%d." % i
            mixer = lambda h: getattr(self, layer["type"])(h, p + "mix.", layer["mixer"], i)  # noqa: E731
            ff = lambda h: self.feed_forward(h, p + "mlp.", layer["mlp"])  # noqa: E731
            if arch == "Lufazen":
                x = x + norm(p + "norm1", mixer(x)) * w(p + "ls1")
                x = x + norm(p + "norm2", ff(x)) * w(p + "ls2")
            elif arch == "Fofapel":
                x = norm(p + "norm1", cfg["postln_alpha"] * x + mixer(x))
                x = norm(p + "norm2", cfg["postln_alpha"] * x + ff(x))
            elif arch == "Gesutar":
                x = x + mixer(norm(p + "norm1", x))
                x = x + ff(norm(p + "norm2", x))
            elif arch == "Mogutar":
                x = x + norm(p + "norm1", mixer(x))
                x = x + norm(p + "norm2", ff(x))
                n = cfg["token_side"]["dim"]
                side = self.table_rows("side.embed", self.tokens, slice(i * n, (i + 1) * n))
                x = x + norm(p + "side.norm", (gelu(x @ w(p + "side.gate").T) * side) @ w(p + "side.proj").T)
            else:
                x = x + m * norm(p + "norm1b", mixer(norm(p + "norm1", x)))
                x = x + m * norm(p + "norm2b", ff(norm(p + "norm2", x)))
        y = norm("final.norm", x[rows]) @ w("embed" if arch == "Vevapel" else "head").T
        cap = cfg.get("logit_softcap")
        return cap * torch.tanh(y / cap) if cap else y


def exact(c, seed):
    cfg = MODELS[c["model"]]
    to = successor(cfg).tolist()
    sequences, tokens = [], []
    for p in prompts_of(c, seed):
        got = [to[p[-1]]]
        while len(got) < c["new"]:
            got.append(to[got[-1]])
        tokens.append(got)
        sequences.append(p + got[:c["new"]])
    _, first = schedule(c)
    ends, at = [], 0
    for s in sequences:
        at += len(s)
        ends.append(at - 1)
    rows = torch.tensor([e for e, f in zip(ends, first) if f == max(first)], device=DEVICE)
    return {"tokens": torch.tensor(tokens), "logits": Plain(cfg, getattr(torch, c["dtype"]), sequences).logits(rows)}
