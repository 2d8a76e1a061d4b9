"""What this framework's users have it compute, as measurable cases.

Each case is one pass through the public entry points on the GPU: the sampler and the
speculative acceptance (`sample_next`, `ops.sample_rows`, `ops.spec_accept`), the
delta-rule seam, one Gated DeltaNet layer, one gated attention layer, one MLP, the MTP
head with its lm_head, and whole forwards (prefill and verify) of a hybrid decoder.
Sizes are those of the repository's own configurations (`tiny_config_dict`,
`dense_8b_config_dict`, its whole models cut to 4 layers -- one period of the 3:1
GDN : attention schedule) and of its benchmark.

`listed()` gives the named cases, `draw(rng)` more of the same ranges; `prepare` makes
inputs, weights and caches on the device from the seed, `run` is the pass, `work` its
unavoidable bytes and flops, `exact` its result in 64-bit torch.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from lollm_amd import ops
from lollm_amd.generate import sample_next
from lollm_amd.qwen3_5 import load
from lollm_amd.qwen3_5.blocks import MLP, GatedAttention, GatedDeltaNet, rope_inv_freq
from lollm_amd.qwen3_5.config import Qwen3_5Config, dense_8b_config_dict, tiny_config_dict
from lollm_amd.qwen3_5.kv import Qwen3_5Cache
from lollm_amd.qwen3_5.mtp import load_mtp
from lollm_amd.qwen3_5.random_init import random_weights

DEV = "cuda"
VOCAB = 151936


# ------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------
def listed():
    return [
        # the reference loop's sampler: one row of logits, the penalty over the context so
        # far, temperature / top-k / top-p at generate()'s defaults; one token to the host
        {"name": "sample one row", "kind": "sample", "rows": 1, "vocab": VOCAB, "context": 517,
         "temperature": 0.7, "top_k": 20, "top_p": 0.8, "penalty": 1.1},
        # acceptance of a serving batch whose drafts were sampled from the MTP head
        {"name": "accept 64x3", "kind": "accept", "batch": 64, "k": 3, "vocab": VOCAB,
         "temperature": 0.7, "top_k": 0, "top_p": 0.95, "sampled": True},
        # the bare delta-rule seam over a verify block
        {"name": "delta rule 8x3", "kind": "rule", "batch": 8, "T": 3, "qk_heads": 16, "v_heads": 32,
         "dtype": "bf16", "l2norm": False},
        # one GDN layer of the verify pass: a batch at different accepted lengths
        {"name": "gdn verify 16x4", "kind": "gdn", "config": "8b", "batch": 16, "T": 4, "fresh": False},
        # one GDN layer over one user's prompt
        {"name": "gdn prefill 1x1847", "kind": "gdn", "config": "8b", "batch": 1, "T": 1847, "fresh": True},
        # one attention layer of the verify pass: long contexts of very different lengths
        {"name": "attn verify 8x4 ragged", "kind": "attn", "config": "8b", "batch": 8, "T": 4,
         "context": 1000, "context_max": 32000},
        # one attention layer over two prompts
        {"name": "attn prefill 2x1999", "kind": "attn", "config": "8b", "batch": 2, "T": 1999,
         "context": 0, "context_max": 0},
        # one MLP over the 64 rows of a 16 x (1 + 3) verify block
        {"name": "mlp 64 rows", "kind": "mlp", "config": "8b", "rows": 64},
        # one draft of 16 sequences: the MTP head and the lm_head
        {"name": "mtp draft 16x1", "kind": "mtp", "config": "8b", "batch": 16, "L": 1, "vocab": VOCAB},
        # the smallest whole call: one user, the tiny model, one new token
        {"name": "tiny decode 1x1", "kind": "model", "config": "tiny", "batch": 1, "T": 1, "context": 131},
        # the verify pass of the benchmark's step (4 of its layers), logits of all rows
        {"name": "verify 16x4", "kind": "model", "config": "8b", "batch": 16, "T": 4, "context": 2048},
        # three prompts through 4 layers, logits of the last position
        {"name": "prefill 3x1500", "kind": "model", "config": "8b", "batch": 3, "T": 1500, "context": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "accept", "rule", "gdn", "gdn", "attn", "attn", "mlp", "mtp", "model"])
    cfg = rng.choice(["8b", "8b", "tiny"])
    if kind == "sample":
        return {"kind": kind, "rows": rng.choice([1, 1, _log(rng, 2, 64)]),
                "vocab": rng.choice([32768, VOCAB]), "context": _log(rng, 16, 4096),
                "temperature": rng.choice([0.0, 0.6, 0.7, 1.0]), "top_k": rng.choice([0, 20, 50]),
                "top_p": rng.choice([0.8, 0.95, 1.0]), "penalty": rng.choice([1.0, 1.05, 1.1])}
    if kind == "accept":
        return {"kind": kind, "batch": _log(rng, 1, 64), "k": rng.randint(1, 3),
                "vocab": rng.choice([32768, VOCAB]), "temperature": rng.choice([0.0, 0.7, 1.0]),
                "top_k": rng.choice([0, 20]), "top_p": rng.choice([0.8, 0.95]),
                "sampled": rng.random() < 0.5}
    if kind == "rule":
        hk = rng.choice([8, 16])
        return {"kind": kind, "batch": _log(rng, 1, 32), "T": rng.randint(1, 6), "qk_heads": hk,
                "v_heads": 2 * hk, "dtype": rng.choice(["bf16", "fp32"]), "l2norm": rng.random() < 0.5}
    if kind == "gdn":
        if rng.random() < 0.5:
            return {"kind": kind, "config": cfg, "batch": _log(rng, 1, 32), "T": rng.randint(1, 4),
                    "fresh": False}
        T = _log(rng, 16, 4096)
        return {"kind": kind, "config": cfg, "batch": _log(rng, 1, max(1, 8192 // T)), "T": T,
                "fresh": rng.random() < 0.6}
    if kind == "attn":
        if rng.random() < 0.5:
            lo = _log(rng, 100, 8000)
            return {"kind": kind, "config": cfg, "batch": _log(rng, 1, 16), "T": rng.randint(1, 4),
                    "context": lo, "context_max": _log(rng, lo, 16000)}
        T = _log(rng, 16, 4096)
        ctx = rng.choice([0, 0, _log(rng, 100, 8000)])
        return {"kind": kind, "config": cfg, "batch": _log(rng, 1, max(1, 4096 // T)), "T": T,
                "context": ctx, "context_max": ctx}
    if kind == "mlp":
        return {"kind": kind, "config": cfg, "rows": _log(rng, 1, 2048)}
    if kind == "mtp":
        return {"kind": kind, "config": cfg, "batch": _log(rng, 1, 32), "L": rng.choice([1, 1, 2, 3]),
                "vocab": rng.choice([32768, VOCAB])}
    if rng.random() < 0.5:
        return {"kind": kind, "config": cfg, "batch": _log(rng, 1, 16), "T": rng.randint(1, 4),
                "context": _log(rng, 100, 2048)}
    T = _log(rng, 16, 2048)
    return {"kind": kind, "config": cfg, "batch": _log(rng, 1, max(1, 4096 // T)), "T": T, "context": 0}


# ------------------------------------------------------------------------------------
# inputs, weights and caches
# ------------------------------------------------------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _raw(config, layer_types=None, vocab=None):
    raw = dense_8b_config_dict() if config == "8b" else tiny_config_dict()
    raw["layer_types"] = layer_types or ["linear_attention"] * 3 + ["full_attention"]
    raw["num_hidden_layers"] = len(raw["layer_types"])
    if vocab:
        raw["vocab_size"] = vocab
    return raw


def _randn(g, *shape, scale=1.0):
    return (scale * torch.randn(*shape, device=DEV, generator=g)).bfloat16()


def _logits(g, *shape):
    """Rows as a language model gives them: a broad bulk and a few tokens well above it."""
    x = 2.5 * torch.randn(*shape, device=DEV, generator=g)
    top = torch.randint(0, shape[-1], (*shape[:-1], 24), device=DEV, generator=g)
    return x.scatter_add(-1, top, 8.0 * torch.rand(*top.shape, device=DEV, generator=g)).bfloat16()


def _layer(c, seed, kind):
    """(config, weights of one layer of that kind, name prefix)."""
    cfg = Qwen3_5Config.from_hf(_raw(c["config"], [kind], vocab=256))
    W = random_weights(cfg, seed, torch.bfloat16, DEV, with_mtp=False)
    return cfg, W, "model.language_model.layers.0."


def _weights(cfg, seed, with_mtp=False):
    """Random weights of a whole model with the residual stream at a trained model's
    proportions: embeddings at the scale of the layers' outputs, and the projections into
    the stream scaled down (as a depth-scaled initialisation does), so that one rounding
    in the first layer is not the whole stream's for all that follow."""
    W = random_weights(cfg, seed, torch.bfloat16, DEV, with_mtp=with_mtp)
    W["model.language_model.embed_tokens.weight"] *= 25
    for name in W:
        if name.endswith(("out_proj.weight", "o_proj.weight", "down_proj.weight")):
            W[name] *= 0.25
    return W


def _inputs(c, seed):
    g, kind = _gen(seed), c["kind"]
    if kind == "sample":
        return {"logits": _logits(g, c["rows"], c["vocab"]),
                "context": torch.randint(0, c["vocab"], (c["rows"], c["context"]), device=DEV,
                                         generator=g, dtype=torch.int32)}
    if kind == "accept":
        B, k, V = c["batch"], c["k"], c["vocab"]
        target = _logits(g, B, k + 1, V)
        # the MTP head's logits are near the target's
        draft = (target[:, :k].float() + 0.7 * torch.randn(B, k, V, device=DEV, generator=g)).bfloat16()
        return {"target": target, "draft": draft}
    if kind == "rule":
        B, T, Hk, Hv, D = c["batch"], c["T"], c["qk_heads"], c["v_heads"], 128
        dt = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
        q, k = (torch.randn(B, T, Hk, D, device=DEV, generator=g) for _ in range(2))
        if not c["l2norm"]:
            q, k = F.normalize(q, dim=-1), F.normalize(k, dim=-1)
        return {"q": q.to(dt), "k": k.to(dt),
                "v": torch.randn(B, T, Hv, D, device=DEV, generator=g).to(dt),
                "g": -F.softplus(torch.randn(B, T, Hv, device=DEV, generator=g)),
                "beta": torch.sigmoid(torch.randn(B, T, Hv, device=DEV, generator=g)).to(dt),
                "state": 0.02 * torch.randn(B, Hv, D, D, device=DEV, generator=g)}
    if kind == "gdn":
        cfg, W, p = _layer(c, seed, "linear_attention")
        B, T = c["batch"], c["T"]
        s = {"cfg": cfg, "W": W, "p": p + "linear_attn.", "x": _randn(g, B, T, cfg.hidden_size)}
        if not c["fresh"]:
            s["conv"] = _randn(g, B, cfg.conv_dim, cfg.linear_conv_kernel_dim - 1)
            s["rec"] = 0.05 * torch.randn(B, cfg.linear_num_value_heads, 128, 128, device=DEV, generator=g)
            if T <= 4:      # a verify pass follows another one: 1 .. 4 of its positions were kept
                s["before"] = _randn(g, B, 4, cfg.hidden_size)
                s["kept"] = torch.randint(0, 4, (B,), device=DEV, generator=g)
        return s
    if kind == "attn":
        cfg, W, p = _layer(c, seed, "full_attention")
        B, T = c["batch"], c["T"]
        lengths = torch.randint(c["context"], c["context_max"] + 1, (B,), device=DEV, generator=g,
                                dtype=torch.int32)
        shape = (B, cfg.num_key_value_heads, c["context_max"] + T, cfg.head_dim)
        return {"cfg": cfg, "W": W, "p": p + "self_attn.", "x": _randn(g, B, T, cfg.hidden_size),
                "lengths": lengths, "k": _randn(g, *shape), "v": _randn(g, *shape, scale=0.5)}
    if kind == "mlp":
        cfg, W, p = _layer(c, seed, "full_attention")
        return {"cfg": cfg, "W": W, "p": p + "mlp.", "x": _randn(g, c["rows"], cfg.hidden_size)}
    if kind == "mtp":
        raw = _raw(c["config"], ["full_attention"], vocab=c["vocab"])
        cfg = Qwen3_5Config.from_hf(raw)
        return {"raw": raw, "cfg": cfg, "W": _weights(cfg, seed, with_mtp=True),
                "hidden": _randn(g, c["batch"], c["L"], cfg.hidden_size),
                "ids": torch.randint(0, c["vocab"], (c["batch"], c["L"]), device=DEV, generator=g)}
    raw = _raw(c["config"])
    cfg = Qwen3_5Config.from_hf(raw)
    return {"raw": raw, "cfg": cfg, "W": _weights(cfg, seed),
            "ids": torch.randint(0, cfg.vocab_size, (c["batch"], c["context"] + c["T"]), device=DEV,
                                 generator=g)}


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    s["case"], s["seed"] = c, int(seed)
    if kind == "sample" and c["rows"] == 1:
        s["context"] = s["context"][0].tolist()
    elif kind == "sample" and c["penalty"] != 1.0:
        s["seen"] = ops.seen_mark(ops.new_seen(c["rows"], c["vocab"], DEV), s["context"], c["vocab"])
    elif kind == "accept":
        pick = c["temperature"] if c["sampled"] else 0.0
        s["drafts"] = torch.stack(
            [ops.sample_rows(s["draft"][:, i].contiguous(), pick, c["top_k"], c["top_p"], 7, 0,
                             slot=c["k"] + 1 + i) for i in range(c["k"])], 1)
        if not c["sampled"] or c["temperature"] <= 0:
            s["draft"] = None
    elif kind == "gdn":
        cfg, B, T = s["cfg"], c["batch"], c["T"]
        s["layer"] = GatedDeltaNet(cfg, s.pop("W"), s["p"])
        s["cache"] = Qwen3_5Cache(cfg, B, T + 16, spec_slots=4)
        if not c["fresh"]:
            s["cache"].set_linear_state(0, s["conv"], s["rec"])
            if "before" in s:
                s["layer"](s["before"], s["cache"], 0)
                s["cache"].commit_all(4)
                s["cache"].rollback(s["kept"])
    elif kind == "attn":
        cfg = s["cfg"]
        s["layer"] = GatedAttention(cfg, s.pop("W"), s["p"],
                                    rope_inv_freq(cfg.rotary_dim, cfg.rope_theta, DEV))
        s["kv_len"] = s["lengths"] + c["T"]
    elif kind == "mlp":
        W, p = s.pop("W"), s["p"]
        s["layer"] = MLP(W[p + "gate_proj.weight"], W[p + "up_proj.weight"], W[p + "down_proj.weight"])
    elif kind == "mtp":
        W = s.pop("W")
        s["model"] = load(s["raw"], W, "hf")
        s["mtp"] = load_mtp(s["model"], W, "hf")
        s["emb"] = s["model"].model.embed_tokens(s["ids"])
    elif kind == "model":
        s["model"] = load(s["raw"], s.pop("W"), "hf")
        s["new"] = s["ids"][:, c["context"]:].contiguous()
        if c["context"]:
            s["past"] = s["model"].new_cache(c["batch"], c["context"] + 16)
            s["model"](s["ids"][:, :c["context"]].contiguous(), s["past"], logits="last")
    return s


# ------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "sample":
        if c["rows"] == 1:
            return sample_next(s["logits"], c["temperature"], c["top_k"], c["top_p"], c["penalty"],
                               s["context"], seed=s["seed"], offset=1)
        x = s["logits"]
        if c["penalty"] != 1.0:
            x = ops.repetition_penalty(x.clone(), s["seen"], c["penalty"])
        return ops.sample_rows(x, c["temperature"], c["top_k"], c["top_p"], s["seed"], 1)
    if kind == "accept":
        return ops.spec_accept(s["target"], s["draft"], s["drafts"], c["temperature"], c["top_k"],
                               c["top_p"], s["seed"], 1)
    if kind == "rule":
        return ops.recurrent_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"],
                                              use_qk_l2norm_in_kernel=c["l2norm"])
    if kind == "gdn":
        # not committed, so the same block can be run again (as a rejected verify is): the
        # new recurrent state or its committed copy is in the other half of `rec`
        out = s["layer"](s["x"], s["cache"], 0)
        return out, s["cache"].layers[0]["rec"]
    if kind == "attn":
        out = s["layer"](s["x"], s["k"], s["v"], s["lengths"], s["kv_len"])
        return out, s["k"], s["v"]
    if kind == "mlp":
        return s["layer"](s["x"])
    if kind == "mtp":
        normed = s["mtp"](s["hidden"], s["emb"])
        return normed, s["model"].lm_head(normed)
    model = s["model"]
    if c["context"]:
        # the verify pass as a decoder runs it before it knows what to commit
        hidden, normed = model.hidden_states(s["new"], s["past"])
        return model.lm_head(normed), hidden
    logits, past, hidden = model(s["new"], model.new_cache(c["batch"], c["T"] + 16), return_hidden=True,
                                 logits="last")
    return logits, hidden


# ------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------
def _gdn_work(cfg, B, T, fresh):
    H, C, Vd, Hv = cfg.hidden_size, cfg.conv_dim, cfg.value_dim, cfg.linear_num_value_heads
    P = C + Vd + 2 * Hv
    state = B * Hv * 128 * 128 * 4
    return {"bytes": 2 * (P * H + H * Vd) + 2 * B * T * H * 2 + (1 if fresh else 2) * state,
            "flops": 2 * B * T * (P * H + H * Vd) + B * T * Hv * 128 * 128 * 6}


def _attn_work(cfg, B, T, keys, pairs):
    """keys: cached keys over the batch; pairs: (query, key) pairs of one head."""
    H, Hq, Hkv, D = cfg.hidden_size, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    w = H * (2 * Hq * D + 2 * Hkv * D) + Hq * D * H
    return {"bytes": 2 * w + 2 * B * T * H * 2 + (keys + 2 * B * T) * Hkv * D * 2 * 2,
            "flops": 2 * B * T * w + 4 * D * Hq * pairs}


def _mlp_work(cfg, rows):
    w = 3 * cfg.hidden_size * cfg.intermediate_size
    return {"bytes": 2 * w + 2 * rows * cfg.hidden_size * 2, "flops": 2 * rows * w}


def _sum(*parts):
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def work(case):
    c = case
    kind = c["kind"]
    if kind == "sample":
        return {"bytes": c["rows"] * c["vocab"] * 2, "flops": 0}
    if kind == "accept":
        rows = c["k"] + 1 + (c["k"] if c["sampled"] and c["temperature"] > 0 else 0)
        return {"bytes": c["batch"] * rows * c["vocab"] * 2, "flops": 0}
    if kind == "rule":
        B, T, Hk, Hv = c["batch"], c["T"], c["qk_heads"], c["v_heads"]
        e = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": 2 * B * Hv * 128 * 128 * 4 + B * T * (2 * Hk + 2 * Hv) * 128 * e,
                "flops": 8 * B * T * Hv * 128 * 128}
    if kind == "mtp":
        cfg = Qwen3_5Config.from_hf(_raw(c["config"], vocab=c["vocab"]))
        B, L, H = c["batch"], c["L"], cfg.hidden_size
        own = 2 * H * H + c["vocab"] * H
        return _sum(_attn_work(cfg, B, L, 0, B * L * (L + 1) // 2), _mlp_work(cfg, B * L),
                    {"bytes": 2 * own + 2 * B * L * c["vocab"], "flops": 2 * B * L * own})
    cfg = Qwen3_5Config.from_hf(_raw(c["config"]))
    if kind == "gdn":
        return _gdn_work(cfg, c["batch"], c["T"], c["fresh"])
    if kind == "mlp":
        return _mlp_work(cfg, c["rows"])
    B, T = c["batch"], c["T"]
    mean = (c["context"] + c.get("context_max", c["context"])) / 2
    attn = _attn_work(cfg, B, T, B * mean, B * (T * mean + T * (T + 1) / 2))
    if kind == "attn":
        return attn
    heads = T if c["context"] else 1
    head = {"bytes": 2 * cfg.vocab_size * (cfg.hidden_size + B * heads),
            "flops": 2 * B * heads * cfg.vocab_size * cfg.hidden_size}
    return _sum(attn, head, *[_gdn_work(cfg, B, T, not c["context"]) for _ in range(3)],
                *[_mlp_work(cfg, B * T) for _ in range(4)])


def tolerance(case):
    """Tokens are exact (the sampler's arithmetic is integer).  The rest: about four times
    the distance measured between the path and `exact` (in the comments), which is what
    bf16 weights, activations and caches leave (fp32 for the seam in fp32)."""
    kind = case["kind"]
    if kind in ("sample", "accept"):
        return "exact"
    if kind == "rule" and case["dtype"] == "fp32":
        rel = 1e-6          # 1e-7 away
    else:
        rel = {"rule": 7e-3,     # 0.0017 away
               "mlp": 1.6e-2,    # 0.0039
               "attn": 1.8e-2,   # 0.0045
               "gdn": 2.5e-2,    # 0.0064
               "mtp": 2e-2,      # 0.0044
               "model": 3e-2,    # 0.012
               }[kind]
    return {"rel": rel, "max": 20 * rel}


# ------------------------------------------------------------------------------------
# the same in 64 bits
# ------------------------------------------------------------------------------------
def _mm(x, w):
    return x.double() @ w.double().t()


def _norm(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * (1 + w.double())


def _delta(q, k, v, g, beta, S, out, t):
    """One position of the gated delta rule; q, k (B, H, D) at the v-heads."""
    S = S * g.exp()[..., None, None]
    d = (v - (S * k[..., None]).sum(-2)) * beta[..., None]
    S = S + k[..., None] * d[..., None, :]
    if out is not None:
        out[:, t] = (S * q[..., None]).sum(-2)
    return S


def _exact_gdn(cfg, W, p, x, conv=None, S=None, keep=None):
    """A GDN layer over x (B, T, H) in 64 bits from a conv state (B, C, K-1) and S.  With
    keep, only the first keep[b] + 1 positions count and (conv, S) after them come back;
    else (out, S)."""
    B, T, _ = x.shape
    Hk, Hv, D, K = cfg.linear_num_key_heads, cfg.linear_num_value_heads, 128, cfg.linear_conv_kernel_dim
    raw = _mm(x, W[p + "in_proj_qkv.weight"])
    if conv is None:
        conv = torch.zeros(B, cfg.conv_dim, K - 1, device=x.device)
    rows = torch.cat([conv.double().transpose(1, 2), raw], 1)
    w = W[p + "conv1d.weight"].reshape(cfg.conv_dim, K).double()
    act = F.silu(sum(rows[:, i:i + T] * w[:, i] for i in range(K)))
    q, k, v = (t.reshape(B, T, -1, D) for t in act.split([cfg.key_dim, cfg.key_dim, cfg.value_dim], -1))
    q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k = (t.repeat_interleave(Hv // Hk, 2) for t in (q, k))
    beta = torch.sigmoid(_mm(x, W[p + "in_proj_b.weight"]))
    g = -W[p + "A_log"].double().exp() * F.softplus(_mm(x, W[p + "in_proj_a.weight"]) + W[p + "dt_bias"].double())
    S = torch.zeros(B, Hv, D, D, device=x.device, dtype=torch.float64) if S is None else S.double()
    out = torch.empty(B, T, Hv, D, device=x.device, dtype=torch.float64)
    for t in range(T):
        S1 = _delta(q[:, t] * D ** -0.5, k[:, t], v[:, t], g[:, t], beta[:, t], S, out, t)
        S = S1 if keep is None else torch.where((t <= keep)[:, None, None, None], S1, S)
    if keep is not None:
        at = keep[:, None] + 1 + torch.arange(K - 1, device=x.device)
        return rows[torch.arange(B, device=x.device)[:, None], at].transpose(1, 2), S
    z = _mm(x, W[p + "in_proj_z.weight"]).reshape(B, T, Hv, D)
    o = out * torch.rsqrt(out.square().mean(-1, keepdim=True) + cfg.rms_norm_eps)
    o = o * W[p + "norm.weight"].double() * F.silu(z)
    return _mm(o.reshape(B, T, -1), W[p + "out_proj.weight"]), S


def _rope(cfg, x, pos):
    """x (B, T, heads, D), pos (B, T); the angles as the model defines them, in fp32."""
    rd = cfg.rotary_dim
    a = (pos.float()[..., None] * rope_inv_freq(rd, cfg.rope_theta, x.device)).double()[:, :, None]
    cos, sin = torch.cat([a, a], -1).cos(), torch.cat([a, a], -1).sin()
    r = x[..., :rd]
    turned = torch.cat([-r[..., rd // 2:], r[..., :rd // 2]], -1)
    return torch.cat([r * cos + turned * sin, x[..., rd:]], -1)


def _exact_attn(cfg, W, p, x, kc=None, vc=None, lengths=None, first=0):
    """(out, new k rows, new v rows) of a gated attention layer; kc / vc (B, Hkv, n, D)."""
    B, T, _ = x.shape
    Hq, Hkv, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    if lengths is None:
        lengths = torch.zeros(B, device=x.device, dtype=torch.int32)
    pos = lengths.long()[:, None] + first + torch.arange(T, device=x.device)
    qg = _mm(x, W[p + "q_proj.weight"]).reshape(B, T, Hq, 2 * D)
    q = _rope(cfg, _norm(qg[..., :D], W[p + "q_norm.weight"], cfg.rms_norm_eps), pos)
    k = _mm(x, W[p + "k_proj.weight"]).reshape(B, T, Hkv, D)
    k = _rope(cfg, _norm(k, W[p + "k_norm.weight"], cfg.rms_norm_eps), pos).transpose(1, 2)
    v = _mm(x, W[p + "v_proj.weight"]).reshape(B, T, Hkv, D).transpose(1, 2)
    o = torch.empty(B, T, Hq, D, device=x.device, dtype=torch.float64)
    rep = Hq // Hkv
    for b in range(B):
        L = int(lengths[b])
        mask = torch.arange(L + T, device=x.device)[None] <= (L + torch.arange(T, device=x.device))[:, None]
        for h in range(Hkv):
            kk, vv = k[b, h], v[b, h]
            if L:
                kk, vv = torch.cat([kc[b, h, :L].double(), kk]), torch.cat([vc[b, h, :L].double(), vv])
            for r in range(rep):
                sc = (q[b, :, h * rep + r] @ kk.t()) * D ** -0.5
                o[b, :, h * rep + r] = sc.masked_fill(~mask, -math.inf).softmax(-1) @ vv
    o = o * torch.sigmoid(qg[..., D:])
    return _mm(o.reshape(B, T, -1), W[p + "o_proj.weight"]), k, v


def _exact_mlp(W, p, x):
    return _mm(F.silu(_mm(x, W[p + "gate_proj.weight"])) * _mm(x, W[p + "up_proj.weight"]),
               W[p + "down_proj.weight"])


def _exact_layer(cfg, W, p, x, kind, first=0):
    h = _norm(x, W[p + "input_layernorm.weight"], cfg.rms_norm_eps)
    if kind == "full_attention":
        x = x + _exact_attn(cfg, W, p + "self_attn.", h, first=first)[0]
    else:
        x = x + _exact_gdn(cfg, W, p + "linear_attn.", h)[0]
    return x + _exact_mlp(W, p + "mlp.", _norm(x, W[p + "post_attention_layernorm.weight"], cfg.rms_norm_eps))


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("sample", "accept"):
        return None
    s = _inputs(case, seed)
    if kind == "rule":
        q, k, v, g, beta = (s[n].double() for n in ("q", "k", "v", "g", "beta"))
        if c["l2norm"]:
            q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = (t.repeat_interleave(c["v_heads"] // c["qk_heads"], 2) for t in (q, k))
        out, S = torch.empty_like(v), s["state"].double()
        for t in range(c["T"]):
            S = _delta(q[:, t] * 128 ** -0.5, k[:, t], v[:, t], g[:, t], beta[:, t], S, out, t)
        return out, S
    cfg, W = s["cfg"], s["W"]
    if kind == "gdn":
        conv, S = s.get("conv"), s.get("rec")
        rec = torch.zeros(c["batch"], 2, cfg.linear_num_value_heads, 128, 128, device=DEV, dtype=torch.float64)
        if S is not None:
            rec[:, 0] = S
        if "before" in s:
            conv, S = _exact_gdn(cfg, W, s["p"], s["before"], conv, S, keep=s["kept"])
            # the first verify pass copied the state it began from to the other half, which
            # its records follow; this one leaves the state after the kept ones in the first
            rec[:, 1] = rec[:, 0]
            rec[:, 0] = S
        out, S = _exact_gdn(cfg, W, s["p"], s["x"], conv, S)
        if "before" not in s:
            rec[:, 1] = S if c["T"] > 4 else rec[:, 0]
        return out, rec
    if kind == "attn":
        out, k, v = _exact_attn(cfg, W, s["p"], s["x"], s["k"], s["v"], s["lengths"])
        if s["k"].numel() > 50_000_000:
            return out, None, None
        kc, vc = s["k"].double(), s["v"].double()
        for b in range(c["batch"]):
            L = int(s["lengths"][b])
            kc[b, :, L:L + c["T"]], vc[b, :, L:L + c["T"]] = k[b], v[b]
        return out, kc, vc
    if kind == "mlp":
        return _exact_mlp(W, s["p"], s["x"])
    table = W["model.language_model.embed_tokens.weight"]
    if kind == "mtp":
        eps = cfg.rms_norm_eps
        emb = _norm(table[s["ids"]].double(), W["mtp.pre_fc_norm_embedding.weight"], eps)
        hid = _norm(s["hidden"].double(), W["mtp.pre_fc_norm_hidden.weight"], eps)
        x = _mm(torch.cat([emb, hid], -1), W["mtp.fc.weight"])
        x = _exact_layer(cfg, W, "mtp.layers.0.", x, "full_attention", first=1)
        x = _norm(x, W["mtp.norm.weight"], eps)
        return x, _mm(x, table)
    x = table[s["ids"]].double()
    for i in range(cfg.num_hidden_layers):
        x = _exact_layer(cfg, W, f"model.language_model.layers.{i}.", x, cfg.layer_type(i))
    hidden = x[:, c["context"]:]
    last = hidden if c["context"] else hidden[:, -1:]
    return _mm(_norm(last, W["model.language_model.norm.weight"], cfg.rms_norm_eps), table), hidden
