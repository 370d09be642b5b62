"""Performance cases of the shared-dictionary attention framework.

Each case is one call as a program makes it: a module or language-model
forward under ``inference_mode``, or one training step (forward and backward)
of a module or of a stack of blocks.  ``listed()`` holds the cases that are
reported, ``draw()`` more of the same ranges, ``exact()`` the same results in
64-bit plain torch.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "double-attention_amd"))

import double_attention as da  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name: str, kind: str, preset: str, batch: int, length: int, **options) -> dict:
    case = {"kind": kind, "preset": preset, "batch": batch, "length": length, "dtype": "bf16", "causal": True,
            "untied": True, "model_dim": 512, "layers": 1, **options}
    return {"name": name, **case} if name else case


def listed() -> list[dict]:
    return [
        # Inference of one attention layer.
        # A short prompt: a few small launches, latency and host work count.
        _case("infer-short", "infer", "a1", 2, 48),
        # The default layer over an ordinary batch.
        _case("infer-a1", "infer", "a1", 8, 512),
        # Four branches and four mixed maps, 128-wide scores.
        _case("infer-4maps", "infer", "qk4-s4", 8, 1024),
        # 512-wide routing against 1536 atoms (the wide-dictionary presets).
        _case("infer-wide", "infer", "a1-r512-d1536", 4, 2048),
        # Long context: one sequence, the causal staircase dominates.
        _case("infer-long", "infer", "a1", 1, 8192),
        # Odd sizes, fp16, no causal mask (an encoder over ragged batches).
        _case("infer-ragged", "infer", "qk2-s2", 5, 777, dtype="fp16", causal=False),
        # The six-layer tied language model, token ids to logits.
        _case("lm-infer", "lm", "qk2-s2", 64, 64, untied=False, layers=6),
        # Training steps of one attention layer: forward, then backward of a
        # regression loss, gradients of the input and of every parameter.
        _case("train-a1", "train", "a1", 8, 512),
        _case("train-4maps", "train", "qk4-s4", 8, 1024),
        _case("train-wide", "train", "a1-r512-d1536", 4, 2048),
        _case("train-long", "train", "a1", 1, 8192),
        # Two blocks (norms, attention, feed-forward) of the language model's
        # training step at its batch.
        _case("train-stack", "stack", "qk2-s2", 64, 64, untied=False, layers=2),
    ]


# Presets with their (branches, maps, routing width, atoms).
_PRESETS = {
    "a1": (1, 1, 256, 512),
    "a1-d1536": (1, 1, 256, 1536),
    "a1-r512-d512": (1, 1, 512, 512),
    "a1-r512-d1024": (1, 1, 512, 1024),
    "a1-r512-d1536": (1, 1, 512, 1536),
    "a1-silu": (1, 1, 256, 512),
    "a1-no-softmax": (1, 1, 256, 512),
    "qk2-s1": (2, 1, 256, 512),
    "qk1-s2": (1, 2, 256, 512),
    "qk2-s2": (2, 2, 256, 512),
    "qk4-s4": (4, 4, 128, 512),
}


def _log_int(rng, low: int, high: int) -> int:
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    """One more case: lengths and batches spread over their logarithm, any
    preset of the list, both 16-bit types, mostly causal."""

    kind = rng.choice(("infer", "infer", "infer", "train", "train", "lm", "stack"))
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind in ("lm", "stack"):
        # Short training sequences in batches, as the language model takes them.
        length = _log_int(rng, 24, 512)
        batch = _log_int(rng, 1, max(1, 4096 // length))
        preset = rng.choice(("a1", "qk2-s2", "qk4-s4"))
        layers = rng.randint(2, 6) if kind == "lm" else rng.randint(1, 2)
        return _case("", kind, preset, batch, length, dtype=dtype, untied=rng.random() < 0.5, layers=layers)
    preset = rng.choice(tuple(_PRESETS))
    branches, maps, routing_dim, atoms = _PRESETS[preset]
    # At most 8192 tokens and 2^26 scores over all maps, fewer tokens for
    # several branches (their routed rows count as tokens).
    tokens = 8192 // (2 if branches * routing_dim > 512 else 1)
    length = _log_int(rng, 32, tokens // (2 if maps > 1 else 1))
    most = max(1, min(tokens // length, (1 << 26) // (maps * length * length)))
    return _case("", kind, preset, _log_int(rng, 1, most), length, dtype=dtype, causal=rng.random() < 0.8,
                 untied=rng.random() < 0.7, model_dim=rng.choice((512, 512, 512, 256, 384, 768)))


_VOCAB = 2048
_FFN = 1536
_TOPICS = 64


def _config(case: dict):
    return da.experiment_config(case["preset"], backend="hip", untied_dictionary=case["untied"],
                                causal=case["causal"], model_dim=case["model_dim"])


def _settle(layer, centres) -> None:
    """Move a fresh layer's dictionary where training takes it: atoms along
    the directions the projected rows have (a freshly drawn dictionary is
    nearly orthogonal to every row, so all rows route alike and the attention
    is uniform).  Atom j belongs to topic j of the inputs as one of the query
    or key branches sees it; value atoms of one topic lie together."""

    bank = layer.bank
    routing_dim, atoms = bank.raw_key.shape
    weights = torch.stack((layer.query.weight, layer.key.weight)).float()
    rows = weights.view(-1, routing_dim, centres.shape[1]) @ centres.t()
    rows = F.normalize(rows, dim=1).permute(0, 2, 1).reshape(-1, routing_dim)
    where = torch.arange(atoms, device=rows.device) % rows.shape[0]
    bank.raw_key.copy_((rows[where] + 0.5 * torch.randn(atoms, routing_dim) * routing_dim ** -0.5).t())
    if bank.raw_value is not None:
        topics = F.normalize(torch.randn(_TOPICS, routing_dim), dim=1)
        bank.raw_value.copy_((topics[where % _TOPICS] + 0.5 * torch.randn(atoms, routing_dim) * routing_dim ** -0.5).t())


@torch.no_grad()
def _target(case: dict, config, model, x):
    """What a training step regresses on: the output of the same layer (or
    stack) at other temperatures and map weights, and noise.  The gradients of
    those few parameters then have the sign that learning gives them; against
    noise alone they would be sums over all scores that cancel to nothing."""

    p = {name: t.double() for name, t in model.state_dict().items()}
    for name, t in p.items():
        if name.endswith("log_score_scales"):
            p[name] = t + 1.0
        elif name.endswith("map_mix_logits"):
            p[name] = t + torch.linspace(-1.0, 1.0, t.numel(), device=t.device, dtype=t.dtype)
    rows = x.detach().double()
    if case["kind"] == "stack":
        out = _stack64(p, "", case, config, rows)
    else:
        out = _attention64(p, "", case, config, rows, *_bank64(p, "bank.", config.eps))
    spread = 1.0 if case["kind"] == "stack" else 0.3
    return (out + spread * torch.randn(out.shape, device=out.device, dtype=out.dtype)).to(x.dtype)


def prepare(case: dict, seed: int) -> dict:
    dtype = _DTYPES[case["dtype"]]
    config = _config(case)
    batch, length, width = case["batch"], case["length"], case["model_dim"]
    torch.manual_seed(seed)
    with torch.device("cuda"):
        if case["kind"] == "lm":
            model = da.DoubleAttentionLM(_VOCAB, length, config, case["layers"], feedforward_dim=_FFN)
        elif case["kind"] == "stack":
            model = da.DoubleAttentionStack(config, case["layers"], feedforward_dim=_FFN)
        else:
            model = da.SharedDictionaryAttention(config)
        model = model.to(dtype)
        # Map weights and temperatures move apart early in training.
        with torch.no_grad():
            for name, p in model.named_parameters():
                if name.endswith("map_mix_logits") or name.endswith("log_score_scales"):
                    p.add_(0.3 * torch.randn(p.shape).to(dtype))
        state = {"kind": case["kind"], "model": model}
        if case["kind"] == "lm":
            state["ids"] = torch.randint(0, _VOCAB, (batch, length))
        else:
            # What a LayerNorm hands on: unit variance, tokens of a few topics.
            centres = torch.randn(_TOPICS, width)
            x = 0.6 * centres[torch.randint(0, _TOPICS, (batch, length))] + 0.8 * torch.randn(batch, length, width)
            state["x"] = x.to(dtype)
            if case["kind"] != "stack":
                with torch.no_grad():
                    _settle(model, centres)
    if case["kind"] in ("infer", "lm"):
        model.eval()
        for p in model.parameters():
            p.requires_grad_(False)
    else:
        state["x"].requires_grad_(True)
        state["target"] = _target(case, config, model, state["x"])
    return state


def run(state: dict):
    model = state["model"]
    if state["kind"] == "infer":
        with torch.inference_mode():
            return model(state["x"])
    if state["kind"] == "lm":
        with torch.inference_mode():
            return model(state["ids"])[0]
    # A training step on 1/2 |out - target|^2, gradients formed anew.
    x = state["x"]
    x.grad = None
    model.zero_grad(set_to_none=True)
    out = model(x)
    out.backward(out.detach() - state["target"])
    grads = {name.replace(".", "_"): p.grad for name, p in model.named_parameters()}
    return {"out": out.detach(), "x": x.grad, **grads}


def _shape(case: dict) -> tuple[int, int, int, int, int]:
    branches, maps, routing_dim, atoms = _PRESETS[case["preset"]]
    score_dim = routing_dim * (branches // maps if branches > maps else 1)
    return branches, maps, routing_dim, atoms, score_dim


def work(case: dict) -> dict:
    branches, maps, routing_dim, atoms, score_dim = _shape(case)
    batch, length, width, layers = case["batch"], case["length"], case["model_dim"], case["layers"]
    tokens, routed = batch * length, branches * routing_dim
    pairs = length * (length + 1) // 2 if case["causal"] else length * length
    # Projections, the route of Q and K rows, the outer attention, the output.
    flops = 2 * tokens * width * (2 * routed + width) + 4 * 2 * tokens * branches * routing_dim * atoms
    flops += 2 * batch * maps * pairs * (score_dim + width) + 2 * tokens * width * width
    weights = width * (2 * routed + 2 * width)
    bank = routing_dim * atoms * (2 if case["untied"] else 1)
    if case["kind"] in ("lm", "stack"):
        flops = layers * (flops + 4 * tokens * width * _FFN)
        weights = layers * (weights + 2 * width * _FFN)
    weights += bank
    rows = tokens * width
    if case["kind"] == "lm":
        flops += 2 * tokens * width * _VOCAB
        weights += (_VOCAB + length) * width
        return {"bytes": 8 * tokens + 2 * (weights + tokens * _VOCAB), "flops": flops}
    if case["kind"] == "infer":
        return {"bytes": 2 * (2 * rows + weights), "flops": flops}
    # Training: two more products for each one of the forward; x and the
    # target read, the output and dx written, weights read, gradients written.
    return {"bytes": 2 * (4 * rows + 2 * weights), "flops": 3 * flops}


def tolerance(case: dict) -> dict:
    # About four times the distance from exact(): outputs 3e-3 in bf16 and
    # 5e-4 in fp16 for one layer, 6e-3 after six; gradients up to 1e-2 and 2e-3
    # (the normalized dictionary's, where a row's parallel part cancels).
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "lm":
        return {"rel": 2e-2 if bf16 else 4e-3, "max": 0.5}
    if case["kind"] == "infer":
        return {"rel": 1e-2 if bf16 else 2e-3, "max": 0.25}
    return {"rel": 3e-2 if bf16 else 1e-2, "max": 0.9}


# ---- the same results in 64 bits ------------------------------------------


def _attention64(p: dict, prefix: str, case: dict, config, x, key, value):
    branches, maps, routing_dim, _, score_dim = _shape(case)
    batch, length, width = x.shape
    q = x @ p[prefix + "query.weight"].t()
    k = x @ p[prefix + "key.weight"].t()
    v = x @ p[prefix + "value.weight"].t() + p[prefix + "value.bias"]
    rows = torch.stack((q, k)).view(2, batch, length, branches, routing_dim)
    u = F.normalize(rows, dim=-1, eps=config.eps)
    beta = p[prefix + "log_beta"].clamp(math.log(0.05), math.log(64.0)).exp()
    logits = u @ key
    if config.dictionary_activation == "silu":
        logits = 2 * F.silu(logits)
    if config.dictionary_assignment == "silu":
        gain = config.dictionary_silu_gain
        weights = 2 / gain * F.silu(gain * logits)
    else:
        weights = torch.softmax(beta * logits, dim=-1)
    z = F.normalize(weights @ value.t(), dim=-1, eps=config.eps)
    if branches > maps:
        # A map of several branches: their scores' root-mean-square sum.
        group = branches // maps
        z = z.reshape(2, batch, length, maps, group * routing_dim) * group ** -0.25
    elif maps > branches:
        z = z.repeat_interleave(maps // branches, dim=3)
    zq, zk = z.permute(0, 1, 3, 2, 4).contiguous().unbind(0)
    gamma = p[prefix + "log_score_scales"].clamp(math.log(0.25), math.log(1024.0)).exp()
    scores = zq @ zk.transpose(-1, -2).contiguous() * gamma.view(1, -1, 1, 1)
    if case["causal"]:
        above = torch.ones(length, length, dtype=torch.bool, device=x.device).triu(1)
        scores = scores.masked_fill(above, -math.inf)
    out = torch.softmax(scores, dim=-1) @ v[:, None]
    if maps > 1:
        alpha = torch.softmax(p[prefix + "map_mix_logits"], dim=0)
        out = (out * alpha.view(1, -1, 1, 1)).sum(1)
    else:
        out = out[:, 0]
    return out @ p[prefix + "output.weight"].t()


def _bank64(p: dict, prefix: str, eps: float):
    key = F.normalize(p[prefix + "raw_key"], dim=0, eps=eps)
    value = F.normalize(p[prefix + "raw_value"], dim=0, eps=eps) if prefix + "raw_value" in p else key
    return key, value


def _stack64(p: dict, prefix: str, case: dict, config, x):
    key, value = _bank64(p, prefix + "banks.0.", config.eps)
    for i in range(case["layers"]):
        at = f"{prefix}blocks.{i}."
        h = F.layer_norm(x, x.shape[-1:], p[at + "attention_norm.weight"], p[at + "attention_norm.bias"])
        x = x + _attention64(p, at + "attention.", case, config, h, key, value)
        h = F.layer_norm(x, x.shape[-1:], p[at + "feedforward_norm.weight"], p[at + "feedforward_norm.bias"])
        h = F.gelu(h @ p[at + "feedforward.0.weight"].t() + p[at + "feedforward.0.bias"])
        x = x + h @ p[at + "feedforward.2.weight"].t() + p[at + "feedforward.2.bias"]
    return x


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    config = _config(case)
    model = state["model"]
    p = {name: t.detach().double() for name, t in model.state_dict().items()}
    training = case["kind"] in ("train", "stack")
    names = [name for name, _ in model.named_parameters()]
    if training:
        for name in names:
            p[name].requires_grad_(True)
    with torch.set_grad_enabled(training):
        if case["kind"] == "lm":
            x = p["token_embedding.weight"][state["ids"]] + p["position_embedding.weight"][None]
            x = _stack64(p, "stack.", case, config, x)
            x = F.layer_norm(x, x.shape[-1:], p["final_norm.weight"], p["final_norm.bias"])
            return x @ p["token_embedding.weight"].t()
        x = state["x"].detach().double().requires_grad_(training)
        if case["kind"] == "stack":
            out = _stack64(p, "", case, config, x)
        else:
            out = _attention64(p, "", case, config, x, *_bank64(p, "bank.", config.eps))
    if not training:
        return out
    out.backward(out.detach() - state["target"].double())
    # The few temperatures and mix logits are single sums over all scores:
    # their error is one draw of the rounding noise, no measure of precision.
    grads = {name.replace(".", "_"): None if p[name].numel() <= 4 else p[name].grad for name in names}
    return {"out": out.detach(), "x": x.grad, **grads}
