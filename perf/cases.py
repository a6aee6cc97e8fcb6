"""The work that is timed: single layers and blocks of a Qwen3-shaped decoder, and whole generations.

Every case goes through the package's public entry points the way a serving
program calls them.  The shapes are the Qwen3-4B ones the package is built
for (hidden 2560, MLP 9728, 32 query and 8 key/value heads of 128, vocabulary
151,936); drawn cases also take other widths, head groups and ragged sizes.
"""

import math
import sys

import torch
from torch import nn
from torch.nn import functional as F

from starter_amd import modules
from starter_amd.engine import KEY_ALIGN, Engine
from starter_amd.kernels.decode_fused import add_rms_norm
from starter_amd.kernels.lm_head import lm_head_argmax
from starter_amd.kernels.prefill import prefill_attention, prefill_qkv
from starter_amd.kernels.rmsnorm import rms_norm
from starter_amd.kernels.rotary import rope_tables
from starter_amd.kernels.skinny_gemm import linear_partials, linear_silu_mul
from starter_amd.kernels.small_query_attention import SmallQueryAttention

HEAD = 128
EPS = 1e-6
THETA = 5_000_000.0
SCALE = HEAD ** -0.5
BF16 = torch.bfloat16


def listed():
    hidden, inner, heads, vocab = 2560, 9728, {"q_heads": 32, "kv_heads": 8}, 151936
    return [
        # The smallest call there is: the norm of one decode step at 8 sequences.
        {"name": "norm_8", "kind": "norm", "rows": 8, "hidden": hidden, "add": False},
        # One decoder MLP block of a decode step (gate/up + SiLU, down, residual
        # add + next norm): one sequence, a ragged batch, a full batch.
        {"name": "mlp_1", "kind": "mlp", "rows": 1, "hidden": hidden, "inner": inner},
        {"name": "mlp_21", "kind": "mlp", "rows": 21, "hidden": hidden, "inner": inner},
        {"name": "mlp_64", "kind": "mlp", "rows": 64, "hidden": hidden, "inner": inner},
        # One decoder attention block of a decode step (packed Q/K/V projection,
        # head norms + RoPE + cache write + attention, output projection,
        # residual add + norm): few long sequences, many ordinary ones.
        {"name": "attend_4x2081", "kind": "attend", "batch": 4, "keys": 2081, "hidden": hidden, **heads},
        {"name": "attend_64x545", "kind": "attend", "batch": 64, "keys": 545, "hidden": hidden, **heads},
        # The language-model head with the greedy choice, logits kept, at a full batch.
        {"name": "head_64", "kind": "head", "rows": 64, "hidden": hidden, "vocab": vocab},
        # A prompt's attention (head norms + RoPE + cache fill, causal attention):
        # one short ragged prompt, a batch of long ones.
        {"name": "prompt_attention_1x333", "kind": "prompt_attention", "batch": 1, "length": 333, **heads},
        {"name": "prompt_attention_4x2048", "kind": "prompt_attention", "batch": 4, "length": 2048, **heads},
        # The MLP module swapped into a transformers model, on a batch of long prompts.
        {"name": "packed_mlp_8192", "kind": "packed_mlp", "rows": 8192, "hidden": hidden, "inner": inner},
        # Whole generations on a few layers of the real widths: one user, a full batch.
        {"name": "generate_1x512", "kind": "generate", "batch": 1, "length": 512, "new": 16, "layers": 4,
         "hidden": hidden, "inner": inner, "vocab": vocab, **heads},
        {"name": "generate_64x160", "kind": "generate", "batch": 64, "length": 160, "new": 16, "layers": 4,
         "hidden": hidden, "inner": inner, "vocab": vocab, **heads},
    ]


def _log(rng, low, high):
    """A whole number from low to high, even over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("norm", "mlp", "attend", "head", "prompt_attention", "packed_mlp", "generate"))
    hidden = rng.choice((2560, 2560, 1024, 2048, 4096))
    inner = 9728 if hidden == 2560 and rng.random() < 0.5 else 64 * rng.randint(hidden // 32, hidden // 16)
    q_heads, kv_heads = rng.choice(((32, 8), (32, 8), (16, 8), (16, 4), (8, 8)))
    heads = {"q_heads": q_heads, "kv_heads": kv_heads}
    if kind == "norm":
        width = hidden if rng.random() < 0.7 else rng.randint(65, 5120)
        return {"kind": kind, "rows": _log(rng, 1, 8192), "hidden": width, "add": rng.random() < 0.5}
    if kind == "mlp":
        return {"kind": kind, "rows": _log(rng, 1, 64), "hidden": hidden, "inner": inner}
    if kind == "attend":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "batch": batch, "keys": _log(rng, 33, min(8192, 65536 // batch)), "hidden": hidden, **heads}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 64), "hidden": hidden if hidden < 4096 else 2560,
                "vocab": 151936 if rng.random() < 0.5 else 16 * rng.randint(2000, 9496)}
    if kind == "prompt_attention":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "batch": batch, "length": _log(rng, 5, min(4096, 8192 // batch)), **heads}
    if kind == "packed_mlp":
        hidden = min(hidden, 2560)
        return {"kind": kind, "rows": _log(rng, 1, 8192), "hidden": hidden, "inner": min(inner, 9728)}
    batch = _log(rng, 1, 64)
    small = rng.random() < 0.3
    return {"kind": kind, "batch": batch, "length": _log(rng, 7, min(1024, 10240 // batch)), "new": rng.randint(2, 16),
            "layers": rng.randint(2, 4), "hidden": 1024 if small else 2560, "inner": 3072 if small else 9728,
            "vocab": 151936, "q_heads": 16 if small else 32, "kv_heads": 8}


# ---------------------------------------------------------------- inputs

class _Maker:
    """Seeded tensors on the GPU, in the order asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, mean=0.0, std=1.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return x.mul_(std).add_(mean).to(BF16)

    def gain(self, width):
        return self.normal(width, mean=1.0, std=0.1)


def _weight_shapes(case):
    """(name, shape, standard deviation) of every parameter of the generated model; 0 is a norm's gain.

    The branches that feed the residual stream are small next to the
    embedding, as in a trained model's first layers, and the head is tied to
    the embedding: the greedy choice is then clear, and one rounding does
    not turn into another text.
    """
    hidden, inner, q, kv = case["hidden"], case["inner"], case["q_heads"] * HEAD, case["kv_heads"] * HEAD
    shapes = [("model.embed_tokens.weight", (case["vocab"], hidden), 0.05), ("model.norm.weight", (hidden,), 0)]
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        shapes += [(p + "input_layernorm.weight", (hidden,), 0), (p + "post_attention_layernorm.weight", (hidden,), 0),
                   (p + "self_attn.q_proj.weight", (q, hidden), 0.02), (p + "self_attn.k_proj.weight", (kv, hidden), 0.02),
                   (p + "self_attn.v_proj.weight", (kv, hidden), 0.02), (p + "self_attn.o_proj.weight", (hidden, q), 0.0005),
                   (p + "self_attn.q_norm.weight", (HEAD,), 0), (p + "self_attn.k_norm.weight", (HEAD,), 0),
                   (p + "mlp.gate_proj.weight", (inner, hidden), 0.02), (p + "mlp.up_proj.weight", (inner, hidden), 0.02),
                   (p + "mlp.down_proj.weight", (hidden, inner), 0.0005)]
    return shapes


def _inv_freq():
    return 1.0 / (THETA ** (torch.arange(0, HEAD, 2, dtype=torch.float32) / HEAD))


def _inputs(case, seed):
    """What the case computes on, without this package: tensors on the GPU (a generation's prompt: lists)."""
    m, kind = _Maker(seed), case["kind"]
    if kind == "norm":
        rows, hidden = case["rows"], case["hidden"]
        return {"x": m.normal(rows, hidden, std=2.0), "branch": m.normal(rows, hidden) if case["add"] else None,
                "gain": m.gain(hidden)}
    if kind == "mlp":
        rows, hidden, inner = case["rows"], case["hidden"], case["inner"]
        return {"x": m.normal(rows, hidden), "residual": m.normal(rows, hidden, std=2.0), "gain": m.gain(hidden),
                "gate_up": m.normal(2 * inner, hidden, std=0.02), "down": m.normal(hidden, inner, std=0.02)}
    if kind == "attend":
        batch, hidden, nq, nk = case["batch"], case["hidden"], case["q_heads"], case["kv_heads"]
        cache = (batch, nk, case["keys"], HEAD)
        return {"x": m.normal(batch, hidden), "residual": m.normal(batch, hidden, std=2.0), "gain": m.gain(hidden),
                "qkv": m.normal((nq + 2 * nk) * HEAD, hidden, std=0.02), "o": m.normal(hidden, nq * HEAD, std=0.02),
                "q_gain": m.gain(HEAD), "k_gain": m.gain(HEAD), "keys": m.normal(*cache), "values": m.normal(*cache)}
    if kind == "head":
        # a hidden state that points at one token, as a trained model's does
        weight = m.normal(case["vocab"], case["hidden"], std=0.02)
        at = torch.randint(0, case["vocab"], (case["rows"],), generator=m.g, device="cuda")
        x = (weight[at].float() * 25 + m.normal(case["rows"], case["hidden"]).float() * 0.87).to(BF16)
        return {"x": x, "weight": weight}
    if kind == "prompt_attention":
        batch, length, nq, nk = case["batch"], case["length"], case["q_heads"], case["kv_heads"]
        return {"qkv": m.normal(batch * length, (nq + 2 * nk) * HEAD), "q_gain": m.gain(HEAD), "k_gain": m.gain(HEAD)}
    if kind == "packed_mlp":
        rows, hidden, inner = case["rows"], case["hidden"], case["inner"]
        return {"x": m.normal(1, rows, hidden), "gate": m.normal(inner, hidden, std=0.02),
                "up": m.normal(inner, hidden, std=0.02), "down": m.normal(hidden, inner, std=0.02)}
    weights = {name: m.normal(*shape, std=std) if std else m.gain(*shape) for name, shape, std in _weight_shapes(case)}
    prompt = torch.randint(0, case["vocab"], (case["batch"], case["length"]), generator=m.g, device="cuda")
    return {"weights": weights, "prompt": prompt.tolist()}


def _config(case):
    """The configuration object of the transformers model that the package adapts."""
    Qwen3Config = sys.modules[modules.Qwen3Attention.__module__].Qwen3Config
    return Qwen3Config(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["inner"],
                       num_hidden_layers=case["layers"], num_attention_heads=case["q_heads"],
                       num_key_value_heads=case["kv_heads"], head_dim=HEAD, max_position_embeddings=32768,
                       rope_theta=THETA, rms_norm_eps=EPS, tie_word_embeddings=True)


class _MLP(nn.Module):
    """The three projections and the activation that PackedMLP takes over."""

    def __init__(self, gate, up, down):
        super().__init__()
        for name, weight in (("gate_proj", gate), ("up_proj", up), ("down_proj", down)):
            layer = nn.Linear(weight.shape[1], weight.shape[0], bias=False, device="meta")
            layer.weight = nn.Parameter(weight, requires_grad=False)
            setattr(self, name, layer)
        self.act_fn = nn.SiLU()


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "attend":  # the caches of a running batch, its last slot to be written by this step
        batch, keys, nk = case["batch"], case["keys"], case["kv_heads"]
        s["cos"], s["sin"] = rope_tables(_inv_freq(), keys, device="cuda")
        s["position"] = torch.tensor([keys - 1], device="cuda")
        s["used"] = torch.full((batch * nk,), keys, dtype=torch.int32, device="cuda")
        s["attention"] = SmallQueryAttention(batch, case["q_heads"], nk, keys, "cuda", key_align=KEY_ALIGN)
    elif kind == "prompt_attention":  # fresh caches with room for the answer
        capacity = case["length"] + 32
        s["cos"], s["sin"] = rope_tables(_inv_freq(), capacity, device="cuda")
        cache = (case["batch"], case["kv_heads"], capacity, HEAD)
        s["keys"], s["values"] = (torch.zeros(cache, dtype=BF16, device="cuda") for _ in range(2))
        s["length"] = case["length"]
    elif kind == "packed_mlp":
        s = {"x": s["x"], "module": modules.PackedMLP(_MLP(s["gate"], s["up"], s["down"]))}
    elif kind == "generate":
        engine = Engine(config=_config(case), keep_logits=True)
        with torch.no_grad():
            for name, parameter in engine.model.named_parameters():
                parameter.copy_(s["weights"][name])
        s = {"engine": engine, "prompt": s["prompt"], "new": case["new"]}
    s["kind"] = kind
    return s


@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "norm":
        if s["branch"] is None:
            return rms_norm(s["x"], s["gain"], EPS)
        return add_rms_norm(s["x"], s["branch"], s["gain"], EPS)
    if kind == "mlp":
        hidden = linear_silu_mul(s["x"], s["gate_up"])
        total, normed = add_rms_norm(s["residual"], linear_partials(hidden, s["down"]), s["gain"], EPS)
        return {"hidden": hidden, "total": total, "normed": normed}
    if kind == "attend":
        attended = s["attention"].run_qkv(linear_partials(s["x"], s["qkv"]), s["q_gain"], s["k_gain"], EPS, EPS,
                                          s["cos"], s["sin"], s["position"], s["keys"], s["values"], s["used"], SCALE)
        attended = attended.view(attended.shape[0], -1)
        total, normed = add_rms_norm(s["residual"], linear_partials(attended, s["o"]), s["gain"], EPS)
        return {"attended": attended, "total": total, "normed": normed, "keys": s["keys"], "values": s["values"]}
    if kind == "head":
        tokens, logits = lm_head_argmax(s["x"], s["weight"], logits=True)
        return {"tokens": tokens, "logits": logits}
    if kind == "prompt_attention":
        q = prefill_qkv(s["qkv"], s["q_gain"], s["k_gain"], EPS, EPS, s["cos"], s["sin"], s["keys"], s["values"], s["length"])
        return {"q": q, "out": prefill_attention(q, s["keys"], s["values"], s["length"], SCALE),
                "keys": s["keys"], "values": s["values"]}
    if kind == "packed_mlp":
        return s["module"](s["x"])
    tokens, logits = [], []
    for step in s["engine"].generate(s["prompt"], s["new"]):
        tokens.append(step)
        logits.append(s["engine"].last_logits)
    return {"tokens": torch.tensor(tokens), "logits": logits}


# ---------------------------------------------------------------- accounts

def work(case):
    kind = case["kind"]
    if kind == "norm":
        rows, hidden = case["rows"], case["hidden"]
        return {"bytes": 2 * hidden * (rows * (4 if case["add"] else 2) + 1), "flops": 5 * rows * hidden}
    if kind == "mlp":
        rows, hidden, inner = case["rows"], case["hidden"], case["inner"]
        return {"bytes": 2 * (3 * hidden * inner + hidden + rows * (4 * hidden + inner)), "flops": 6 * rows * hidden * inner}
    if kind == "attend":
        batch, keys, hidden, nq, nk = (case[k] for k in ("batch", "keys", "hidden", "q_heads", "kv_heads"))
        weights = hidden * (2 * nq + 2 * nk) * HEAD
        return {"bytes": 2 * (weights + batch * (2 * nk * keys * HEAD + 4 * hidden + nq * HEAD)),
                "flops": 2 * batch * weights + 4 * batch * nq * keys * HEAD}
    if kind == "head":
        rows, hidden, vocab = case["rows"], case["hidden"], case["vocab"]
        return {"bytes": 2 * (vocab * hidden + rows * (hidden + vocab)), "flops": 2 * rows * hidden * vocab}
    if kind == "prompt_attention":
        batch, length, nq, nk = (case[k] for k in ("batch", "length", "q_heads", "kv_heads"))
        return {"bytes": 2 * batch * length * HEAD * (3 * nq + 4 * nk),
                "flops": 2 * batch * nq * length * (length + 1) * HEAD}
    if kind == "packed_mlp":
        rows, hidden, inner = case["rows"], case["hidden"], case["inner"]
        return {"bytes": 2 * (3 * hidden * inner + 2 * rows * hidden), "flops": 6 * rows * hidden * inner}
    batch, length, new, layers, hidden, inner, vocab, nq, nk = (case[k] for k in (
        "batch", "length", "new", "layers", "hidden", "inner", "vocab", "q_heads", "kv_heads"))
    layer = hidden * (2 * nq + 2 * nk) * HEAD + 3 * hidden * inner
    body, head = layers * layer, hidden * vocab
    cache = sum(length + i for i in range(1, new)) * batch * layers * 2 * nk * HEAD
    steps = new * (body + head + batch * vocab) + cache + batch * length * layers * 2 * nk * HEAD
    tokens = batch * (length + new - 1)
    return {"bytes": 2 * steps, "flops": 2 * (tokens * body + batch * new * head)
            + 2 * batch * nq * HEAD * layers * (length * (length + 1) + 2 * sum(length + i for i in range(1, new)))}


def tolerance(case):
    """About four times what the same roundings differ by when the sums run in another order (library products,
    other key segments, torch's attention): single bf16 results then fall on the other side of a rounding."""
    kind = case["kind"]
    if kind in ("norm", "mlp", "head", "packed_mlp"):  # seen: up to 1.4e-4, single values by one unit (0.0078)
        return {"rel": 1e-3, "max": 0.04}
    if kind in ("attend", "prompt_attention"):  # the weights are rounded against a running maximum: 2.2e-3, 0.016
        return {"rel": 9e-3, "max": 0.06}
    return {"rel": 0.027, "max": 0.2}  # through all layers and steps in 16 bits: 6.8e-3, 0.05


# ---------------------------------------------------------------- 64-bit values

def _norm64(x, gain):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain.double()


def _rope64(x, start):
    """Rotate the halves of x [B, heads, T, 128] by its positions start .. start + T."""
    angle = torch.arange(start, start + x.shape[2], device=x.device).double()[:, None] * _inv_freq().to(x.device).double()
    cos, sin = torch.cat([angle, angle], -1).cos(), torch.cat([angle, angle], -1).sin()
    low, high = x[..., :HEAD // 2], x[..., HEAD // 2:]
    return x * cos + torch.cat([-high, low], -1) * sin


def _heads64(packed, nq, nk, q_gain, k_gain, start):
    """q, k, v [B, heads, T, 128] of packed rows [B, T, (nq + 2 nk) * 128]: head norms and RoPE applied."""
    batch, length = packed.shape[:2]
    q, k, v = packed.view(batch, length, nq + 2 * nk, HEAD).transpose(1, 2).split((nq, nk, nk), 1)
    return _rope64(_norm64(q, q_gain), start), _rope64(_norm64(k, k_gain), start), v


def _attention64(q, k, v, start):
    """Causal attention of queries at positions start .. against the keys from position 0: [B, T, heads * 128]."""
    batch, nq, length, _ = q.shape
    groups = nq // k.shape[1]
    out = torch.empty((batch, length, nq, HEAD), dtype=torch.float64, device=q.device)
    hide = torch.arange(k.shape[2], device=q.device)[None] > torch.arange(start, start + length, device=q.device)[:, None]
    for b in range(batch):
        for h in range(nq):
            p = (q[b, h] @ k[b, h // groups].T).mul_(SCALE).masked_fill_(hide, -math.inf)
            out[b, :, h] = torch.softmax(p, -1) @ v[b, h // groups]
    return out.view(batch, length, nq * HEAD)


def _decode_attention64(q, k, v):
    """One query position q [B, nq, 1, 128] against every key: [B, nq * 128]."""
    batch, nq = q.shape[:2]
    q = q.reshape(batch, k.shape[1], -1, HEAD)
    p = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) * SCALE, -1)
    return torch.matmul(p, v.contiguous()).reshape(batch, nq * HEAD)


def _generate64(case, s):
    w = {name: t.double() for name, t in s["weights"].items()}
    batch, nq, nk = case["batch"], case["q_heads"], case["kv_heads"]
    cache = [None] * case["layers"]
    ids, start, logits = torch.tensor(s["prompt"], device="cuda"), 0, []
    for _ in range(case["new"]):
        x = w["model.embed_tokens.weight"][ids]
        for i in range(case["layers"]):
            p = {name.split(".", 3)[3]: t for name, t in w.items() if name.startswith("model.layers.%d." % i)}
            h = _norm64(x, p["input_layernorm.weight"])
            packed = torch.cat([F.linear(h, p["self_attn.%s_proj.weight" % n]) for n in "qkv"], -1)
            q, k, v = _heads64(packed, nq, nk, p["self_attn.q_norm.weight"], p["self_attn.k_norm.weight"], start)
            if cache[i] is not None:
                k, v = torch.cat([cache[i][0], k], 2), torch.cat([cache[i][1], v], 2)
            cache[i] = (k, v)
            a = _decode_attention64(q, k, v).unsqueeze(1) if start else _attention64(q, k, v, start)
            x = x + F.linear(a, p["self_attn.o_proj.weight"])
            h = _norm64(x, p["post_attention_layernorm.weight"])
            x = x + F.linear(F.silu(F.linear(h, p["mlp.gate_proj.weight"])) * F.linear(h, p["mlp.up_proj.weight"]),
                             p["mlp.down_proj.weight"])
        start += ids.shape[1]
        logits.append(F.linear(_norm64(x[:, -1], w["model.norm.weight"]), w["model.embed_tokens.weight"]))
        ids = logits[-1].argmax(-1, keepdim=True)
    return {"tokens": None, "logits": logits}


@torch.no_grad()
def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "generate":
        return _generate64(case, s)
    d = {k: v.double() for k, v in s.items() if isinstance(v, torch.Tensor)}
    if kind == "norm":
        if not case["add"]:
            return _norm64(d["x"], s["gain"])
        total = d["x"] + d["branch"]
        return total, _norm64(total, s["gain"])
    if kind == "mlp":
        gate, up = F.linear(d["x"], d["gate_up"]).chunk(2, -1)
        hidden = F.silu(gate) * up
        total = d["residual"] + F.linear(hidden, d["down"])
        return {"hidden": hidden, "total": total, "normed": _norm64(total, s["gain"])}
    if kind == "attend":
        nq, nk, last = case["q_heads"], case["kv_heads"], case["keys"] - 1
        q, k, v = _heads64(F.linear(d["x"], d["qkv"]).unsqueeze(1), nq, nk, s["q_gain"], s["k_gain"], last)
        keys, values = d["keys"], d["values"]
        keys[:, :, last], values[:, :, last] = k[:, :, 0], v[:, :, 0]
        attended = _decode_attention64(q, keys, values)
        total = d["residual"] + F.linear(attended, d["o"])
        return {"attended": attended, "total": total, "normed": _norm64(total, s["gain"]), "keys": keys, "values": values}
    if kind == "head":
        return {"tokens": None, "logits": F.linear(d["x"], d["weight"])}
    if kind == "prompt_attention":
        batch, length = case["batch"], case["length"]
        packed = d["qkv"].view(batch, length, -1)
        q, k, v = _heads64(packed, case["q_heads"], case["kv_heads"], s["q_gain"], s["k_gain"], 0)
        keys, values = (torch.zeros((*t.shape[:2], length + 32, HEAD), dtype=torch.float64, device="cuda") for t in (k, v))
        keys[:, :, :length], values[:, :, :length] = k, v
        out = _attention64(q, k, v, 0).view(batch, length, case["q_heads"], HEAD)
        return {"q": q.transpose(1, 2).contiguous(), "out": out, "keys": keys, "values": values}
    hidden = F.silu(F.linear(d["x"], d["gate"])) * F.linear(d["x"], d["up"])
    return F.linear(hidden, d["down"])
