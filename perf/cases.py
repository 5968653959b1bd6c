"""The work a user of gptrig has it do, as cases that can be timed and compared.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass
through the public entry points, ``work`` what the pass cannot do without,
``exact`` the same outputs in 64 bits from plain torch, ``tolerance`` how far
two correct implementations at the same precision may differ.

Imported with the repository's root as the working folder.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpt-speedrun-tpu_amd"))

from gptrig import nn  # noqa: E402
from gptrig.attention import attention_softmax_scale  # noqa: E402
from gptrig.kernels import AttentionConfig, make_causal_attention  # noqa: E402
from gptrig.kernels.linear_cross_entropy import tiled_tied_cross_entropy, tiled_tied_cross_entropy_losses  # noqa: E402
from gptrig.moe import routed_mlp_local  # noqa: E402
from gptrig.optim import OptimizerConfig  # noqa: E402
from gptrig.train import GPTConfig, GPTTrainer  # noqa: E402

DEVICE = "cuda:0"
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
VOCAB = 50304  # storage rows of the embedding; 50257 of them are classes with the GPT-2 tokenizer


def listed() -> list[dict]:
    return [
        # The attention layer of the 125M model at the sizes the benchmark
        # isolates, forward and backward.
        attention("attention-train", batch=16, heads=12, seq=1024, dim=64),
        # Long-context training on packed documents (the 8k window with
        # document masking and the 1/head_dim scale), q/k/v as a program has
        # them after one QKV projection.
        attention("attention-documents-8k", batch=2, heads=12, seq=8192, dim=64, documents=True, packed=True,
                  rule="inverse_head_dim"),
        # Heads of 128 over a window that is no multiple of any tile.
        attention("attention-wide-ragged", batch=4, heads=6, seq=2000, dim=128, packed=True),
        # The smallest call: one short sequence, forward only (evaluating a
        # prompt), where latency and launches count.
        attention("attention-prompt", batch=1, heads=8, seq=129, dim=64, backward=False),
        # The language-model head and its loss in training, through the
        # memory-bounded public call with its default tile.
        loss("loss-train", tokens=16384, width=768),
        # Scoring held-out text: per-token losses without gradients, a token
        # count that is no multiple of a tile, float32 master embedding, 47
        # storage rows that are no classes.
        loss("loss-score", tokens=8 * 1023, width=768, classes=50257, mean=False, backward=False, master=True),
        # The loss with float32 compute, forward and backward.
        loss("loss-float32", tokens=2048, width=512, compute="float32", master=True),
        # The bandwidth-bound passes of one block (norm, rotary embedding of
        # q, GELU), forward and backward, at a training micro-batch.
        passes("block-passes", batch=32, seq=1024, width=768, heads=12, hidden=3072),
        # The routed MLP of the MoE recipe's training step.
        routed("routed-train", batch=32, seq=1024, width=768, experts=8, top_k=2, hidden=1536),
        # The same layer fine-tuned on one short ragged sequence.
        routed("routed-short", batch=1, seq=200, width=512, experts=8, top_k=2, hidden=1024),
        # Whole optimizer steps: the 60M-class model of the smallest training
        # configuration, and the 125M model at the benchmark's batch.
        step("step-60m", layers=8, heads=8, width=512, batch=8, micro=8),
        step("step-125m", layers=12, heads=12, width=768, batch=128, micro=64),
    ]


def attention(name, *, batch, heads, seq, dim, documents=False, packed=False, backward=True,
              rule="inverse_sqrt_head_dim") -> dict:
    return dict(name=name, kind="attention", batch=batch, heads=heads, seq=seq, dim=dim, documents=documents,
                packed=packed, backward=backward, rule=rule)


def loss(name, *, tokens, width, classes=VOCAB, mean=True, backward=True, master=False, compute="bfloat16",
         vocab=VOCAB) -> dict:
    return dict(name=name, kind="loss", tokens=tokens, width=width, vocab=vocab, classes=classes, mean=mean,
                backward=backward, master=master, compute=compute)


def passes(name, *, batch, seq, width, heads, hidden) -> dict:
    return dict(name=name, kind="passes", batch=batch, seq=seq, width=width, heads=heads, hidden=hidden)


def routed(name, *, batch, seq, width, experts, top_k, hidden, backward=True) -> dict:
    return dict(name=name, kind="routed", batch=batch, seq=seq, width=width, experts=experts, top_k=top_k,
                hidden=hidden, backward=backward)


def step(name, *, layers, heads, width, batch, micro, seq=1024, documents=False) -> dict:
    return dict(name=name, kind="step", layers=layers, heads=heads, width=width, batch=batch, micro=micro, seq=seq,
                documents=documents)


def draw(rng) -> dict:
    """One more case of the ranges above; sizes over their logarithm, odd ones among them."""

    def size(low, high, multiple=1):
        n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
        return max(low, n // multiple * multiple)

    kind = rng.choice(["attention", "attention", "loss", "loss", "passes", "routed", "routed", "step"])
    if kind == "attention":
        seq = size(64, 8192)
        dim = rng.choice([64, 64, 64, 96, 128])
        heads = rng.choice([6, 8, 12])
        # up to the scores of the 8k case
        most = max(1, min(64, int(24 * 8192 ** 2 * 64 / (heads * seq ** 2 * dim))))
        case = attention("", batch=size(1, most), heads=heads, seq=seq, dim=dim, documents=rng.random() < 0.4,
                         packed=rng.random() < 0.6, backward=rng.random() < 0.7,
                         rule=rng.choice(["inverse_sqrt_head_dim", "inverse_head_dim"]))
    elif kind == "loss":
        classes = rng.choice([VOCAB, 50257])
        if rng.random() < 0.25:
            case = loss("", tokens=size(128, 2048), width=rng.choice([256, 512, 768]), classes=classes,
                        mean=rng.random() < 0.5, backward=rng.random() < 0.6, master=True, compute="float32")
        else:
            case = loss("", tokens=size(128, 16384), width=rng.choice([512, 576, 768, 1024]), classes=classes,
                        mean=rng.random() < 0.5, backward=rng.random() < 0.6, master=rng.random() < 0.5)
    elif kind == "passes":
        heads = rng.choice([8, 12, 16])
        case = passes("", batch=rng.randint(1, 32), seq=size(64, 1024), width=64 * heads, heads=heads,
                      hidden=256 * heads)
    elif kind == "routed":
        width = rng.choice([256, 512, 768])
        case = routed("", batch=rng.randint(1, 16), seq=size(50, 2048), width=width,
                      experts=rng.choice([4, 8, 16]) if width < 768 else rng.choice([4, 8]),
                      top_k=rng.choice([1, 2]), hidden=width * rng.choice([2, 4]), backward=rng.random() < 0.7)
    else:
        heads, dim = rng.choice([(4, 64), (4, 128), (8, 64), (12, 64), (6, 128)])
        micro = rng.randint(1, 8)
        seq = size(100, 1024)
        while micro * seq % 8:  # the step's token groups
            seq += 1
        case = step("", layers=rng.randint(2, 8), heads=heads, width=heads * dim, batch=micro * rng.choice([1, 2]),
                    micro=micro, seq=seq, documents=rng.random() < 0.3)
    del case["name"]
    return case


# -- inputs ------------------------------------------------------------------------


class _Draws:
    """Seeded draws on the GPU."""

    def __init__(self, seed: int):
        self.gen = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def normal(self, *shape, scale=1.0, dtype=BF16):
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * scale).to(dtype)

    def whole(self, high, *shape, dtype=torch.int32):
        return torch.randint(0, high, shape, generator=self.gen, device=DEVICE, dtype=dtype)


def _document_ids(batch: int, seq: int, seed: int) -> torch.Tensor:
    """Packed documents of 1..3000 tokens; the id counts them along the row."""

    rng = np.random.default_rng(seed)
    ids = np.zeros((batch, seq), np.int32)
    for b in range(batch):
        starts = np.cumsum(rng.integers(1, 3001, size=seq))
        ids[b, starts[starts < seq]] = 1
    return torch.from_numpy(np.cumsum(ids, axis=1, dtype=np.int32)).to(DEVICE)


def _leaf(t: torch.Tensor) -> torch.Tensor:
    return t.detach().requires_grad_()


def prepare(case: dict, seed: int) -> dict:
    state = dict(case)
    rand = _Draws(seed)
    if case["kind"] == "attention":
        B, H, S, D = case["batch"], case["heads"], case["seq"], case["dim"]
        if case["packed"]:  # [B, S, 3, H, D] from the QKV projection; the output's gradient comes as [B, S, H, D]
            qkv = rand.normal(B, S, 3, H, D)
            q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
            do = rand.normal(B, S, H, D).transpose(1, 2)
        else:
            q, k, v, do = (rand.normal(B, H, S, D) for _ in range(4))
        grad = case["backward"]
        state.update(q=_leaf(q) if grad else q, k=_leaf(k) if grad else k, v=_leaf(v) if grad else v, do=do,
                     segments=_document_ids(B, S, seed) if case["documents"] else None,
                     attention=make_causal_attention(
                         AttentionConfig(softmax_scale=attention_softmax_scale(case["rule"], D))))
    elif case["kind"] == "loss":
        n, d, V = case["tokens"], case["width"], case["vocab"]
        f32 = case["compute"] == "float32"
        hidden = rand.normal(n, d, dtype=F32 if f32 else BF16)
        weight = rand.normal(V, d, scale=0.02, dtype=F32 if case["master"] else BF16)
        grad = case["backward"]
        state.update(hidden=_leaf(hidden) if grad else hidden, weight=_leaf(weight) if grad else weight,
                     targets=rand.whole(case["classes"], n), cotangent=rand.normal(n, dtype=F32).abs() / n)
    elif case["kind"] == "passes":
        B, S, d, H, f = case["batch"], case["seq"], case["width"], case["heads"], case["hidden"]
        state.update(x=_leaf(rand.normal(B, S, d)), scale=_leaf(1.0 + rand.normal(d, scale=0.1, dtype=F32)),
                     q=_leaf(rand.normal(B, S, H, d // H)), h=_leaf(rand.normal(B, S, f)), dx=rand.normal(B, S, d),
                     dq=rand.normal(B, S, H, d // H), dh=rand.normal(B, S, f))
    elif case["kind"] == "routed":
        B, S, d, E, f = case["batch"], case["seq"], case["width"], case["experts"], case["hidden"]
        grad = case["backward"]
        tensors = dict(x=rand.normal(B, S, d), router_w=rand.normal(d, E, scale=0.02, dtype=F32),
                       up_w=rand.normal(E, d, f, scale=0.02, dtype=F32),
                       up_b=rand.normal(E, f, scale=0.02, dtype=F32),
                       down_w=rand.normal(E, f, d, scale=0.02, dtype=F32),
                       down_b=rand.normal(E, d, scale=0.02, dtype=F32))
        state["args"] = [_leaf(t) if grad else t for t in tensors.values()]
        state["douts"] = (rand.normal(B, S, d), rand.normal(E, scale=0.1, dtype=F32))
    else:
        config = GPTConfig(layers=case["layers"], heads=case["heads"], d_model=case["width"], vocab_size=VOCAB,
                           semantic_vocab_size=VOCAB, seq_len=case["seq"], batch_size=case["batch"],
                           micro_batch_size=case["micro"], document_masking=case["documents"],
                           optimizer=OptimizerConfig(steps=10000, warmup_steps=2000))
        window = rand.whole(VOCAB, case["batch"], case["seq"] + 1)
        if case["documents"]:  # a boundary token about every 300 tokens
            window[rand.whole(300, *window.shape) == 0] = config.document_boundary_token
        state.update(trainer=GPTTrainer(config, seed=seed), x=window[:, :-1].contiguous(),
                     y=window[:, 1:].contiguous())
    return state


# -- one pass ------------------------------------------------------------------------


def run(state: dict):
    kind = state["kind"]
    if kind == "attention":
        q, k, v = state["q"], state["k"], state["v"]
        o = state["attention"](q, k, v, state["segments"])
        return (o, *torch.autograd.grad(o, (q, k, v), state["do"])) if state["backward"] else o
    if kind == "loss":
        call = tiled_tied_cross_entropy if state["mean"] else tiled_tied_cross_entropy_losses
        hidden, weight = state["hidden"], state["weight"]
        value = call(hidden, weight, state["targets"], semantic_vocab_size=state["classes"],
                     compute_dtype=F32 if state["compute"] == "float32" else BF16)
        if not state["backward"]:
            return value
        return (value, *torch.autograd.grad(value, (hidden, weight), None if state["mean"] else state["cotangent"]))
    if kind == "passes":
        x, scale, q, h = state["x"], state["scale"], state["q"], state["h"]
        y, r, g = nn.rms_norm(x, scale), nn.apply_rotary(q), nn.gelu(h)
        return (y, r, g, *torch.autograd.grad((y, r, g), (x, scale, q, h), (state["dx"], state["dq"], state["dh"])))
    if kind == "routed":
        args = state["args"]
        out, mean_probability, load, summary = routed_mlp_local(*args, experts=state["experts"],
                                                                top_k=state["top_k"])
        if not state["backward"]:
            return out, mean_probability, load, summary
        return (out, mean_probability, load, summary,
                *torch.autograd.grad((out, mean_probability), args, state["douts"]))
    trainer = state["trainer"]
    trainer.train_step(state["x"], state["y"])
    return trainer.loss, trainer.norm, trainer.arena.g, trainer.arena.p


# -- what a pass cannot do without -------------------------------------------------------


def _visible_pairs(case: dict) -> float:
    """Query-key pairs of one head over the batch: causal, and (on average) within a document."""

    S = case["seq"]
    pairs = S * (S + 1) / 2
    if case["documents"]:
        pairs = min(pairs, S * 1000.0)  # documents uniform in 1..3000 tokens: E[n^2] / (2 E[n])
    return case["batch"] * pairs


def work(case: dict) -> dict:
    if case["kind"] == "attention":
        B, H, S, D = case["batch"], case["heads"], case["seq"], case["dim"]
        flops = 4.0 * H * D * _visible_pairs(case)
        size = 2.0 * B * H * S * D
        return {"bytes": (12 if case["backward"] else 4) * size, "flops": flops * (3 if case["backward"] else 1)}
    if case["kind"] == "loss":
        n, d, V = case["tokens"], case["width"], case["vocab"]
        h, w = (4 if case["compute"] == "float32" else 2), (4 if case["master"] else 2)
        moved = n * d * h + V * d * w
        return {"bytes": float(moved * (2 if case["backward"] else 1)),
                "flops": 2.0 * n * d * V * (3 if case["backward"] else 1)}
    if case["kind"] == "passes":
        rows = case["batch"] * case["seq"]
        elements = rows * (2 * case["width"] + case["hidden"])
        return {"bytes": 10.0 * elements, "flops": 0.0}
    if case["kind"] == "routed":
        tokens, d, f, E = case["batch"] * case["seq"], case["width"], case["hidden"], case["experts"]
        flops = 4.0 * tokens * case["top_k"] * d * f
        moved = 4.0 * tokens * d + 8.0 * E * d * f
        return {"bytes": moved * (2 if case["backward"] else 1), "flops": flops * (3 if case["backward"] else 1)}
    L, d, S = case["layers"], case["width"], case["seq"]
    tokens = case["batch"] * S
    parameters = L * 12 * d * d + 2 * VOCAB * d
    flops = tokens * (6.0 * (L * 12 * d * d + VOCAB * d) + 6.0 * L * d * (S + 1))
    return {"bytes": 28.0 * parameters, "flops": flops}


def tolerance(case: dict) -> dict:
    # About four times the distance of a pass from exact().  bf16 results of
    # float32 sums: an ulp is 2^-8, and probabilities and score gradients are
    # rounded to bf16 before their products.
    if case["kind"] == "attention":
        return {"rel": 1.0e-2, "max": 0.3}
    if case["kind"] == "loss":
        if case["compute"] == "float32":
            return {"rel": 4.0e-6, "max": 1.0e-3}
        # Without gradients the outputs are float32 sums of exact products.
        return {"rel": 7.0e-3, "max": 0.3} if case["backward"] else {"rel": 1.0e-6, "max": 2.0e-5}
    if case["kind"] == "passes":
        return {"rel": 8.0e-3, "max": 0.03}
    if case["kind"] == "routed":
        return {"rel": 2.0e-2, "max": 0.8}
    # A whole step: a rounding in one layer travels through all that follow.
    return {"rel": 3.0e-2, "max": 0.95}


# -- the same in 64 bits -----------------------------------------------------------------


def exact(case: dict, seed: int):
    if case["kind"] == "step":
        return None
    state = prepare(case, seed)
    return {"attention": _exact_attention, "loss": _exact_loss, "passes": _exact_passes,
            "routed": _exact_routed}[case["kind"]](state)


def _exact_attention(state: dict):
    B, H, S, D = state["batch"], state["heads"], state["seq"], state["dim"]
    scale = attention_softmax_scale(state["rule"], D)
    q, k, v, do = (state[n].detach() for n in ("q", "k", "v", "do"))
    out = [torch.empty((B, H, S, D), dtype=F64, device=DEVICE) for _ in range(4 if state["backward"] else 1)]
    at = torch.arange(S, device=DEVICE)
    for b in range(B):
        hidden = at[None, :] > at[:, None]
        if state["segments"] is not None:
            ids = state["segments"][b]
            hidden = hidden | (ids[None, :] != ids[:, None])
        for h in range(H):
            qh, kh, vh, gh = (t[b, h].to(F64) for t in (q, k, v, do))
            p = torch.softmax((qh @ kh.T * scale).masked_fill_(hidden, -math.inf), dim=-1)
            o = p @ vh
            out[0][b, h] = o
            if state["backward"]:
                ds = p * (gh @ vh.T - (gh * o).sum(-1, keepdim=True)) * scale
                out[1][b, h], out[2][b, h], out[3][b, h] = ds @ kh, ds.T @ qh, p.T @ gh
    return tuple(out) if state["backward"] else out[0]


def _exact_loss(state: dict):
    n, C = state["tokens"], state["classes"]
    operand = F32 if state["compute"] == "float32" else BF16
    h, w = state["hidden"].detach().to(operand).to(F64), state["weight"].detach().to(operand).to(F64)
    targets = state["targets"].long()
    losses = torch.empty(n, dtype=F64, device=DEVICE)
    dh, dw = torch.zeros_like(h), torch.zeros_like(w)
    cotangent = torch.full((n,), 1.0 / n, dtype=F64, device=DEVICE) if state["mean"] else state["cotangent"].to(F64)
    for i in range(0, n, 2048):
        part, t = h[i:i + 2048], targets[i:i + 2048, None]
        logits = part @ w[:C].T
        lse = torch.logsumexp(logits, dim=-1)
        losses[i:i + 2048] = lse - logits.gather(1, t)[:, 0]
        if state["backward"]:
            g = torch.exp(logits - lse[:, None]) * cotangent[i:i + 2048, None]
            g.scatter_add_(1, t, -cotangent[i:i + 2048, None])
            dh[i:i + 2048] = g @ w[:C]
            dw[:C] += g.T @ part
    value = losses.mean() if state["mean"] else losses
    return (value, dh, dw) if state["backward"] else value


def _exact_passes(state: dict):
    x, scale, q, h = (state[n].detach().to(F64) for n in ("x", "scale", "q", "h"))
    scale = state["scale"].detach().to(BF16).to(F64)
    x, scale, q, h = (t.requires_grad_() for t in (x, scale, q, h))
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1.0e-5) * scale
    D = q.shape[-1]
    rate = 10000.0 ** (-torch.arange(0, D, 2, dtype=F64, device=DEVICE) / D)
    angle = torch.arange(q.shape[1], dtype=F64, device=DEVICE)[:, None] * rate
    c, s = (f(angle).to(BF16).to(F64)[None, :, None, :] for f in (torch.cos, torch.sin))
    even, odd = q[..., 0::2], q[..., 1::2]
    r = torch.stack((even * c - odd * s, even * s + odd * c), dim=-1).reshape(q.shape)
    g = torch.nn.functional.gelu(h, approximate="tanh")
    grads = torch.autograd.grad((y, r, g), (x, scale, q, h), [state[n].to(F64) for n in ("dx", "dq", "dh")])
    return (y.detach(), r.detach(), g.detach(), *grads)


def _exact_routed(state: dict):
    B, S, d, E, k = state["batch"], state["seq"], state["width"], state["experts"], state["top_k"]
    args = [t.detach() for t in state["args"]]
    # The expert matmuls take bfloat16 operands; the router stays float32.
    args = [t.to(F64) if i < 2 else t.to(BF16).to(F64) for i, t in enumerate(args)]
    x, router_w, up_w, up_b, down_w, down_b = (t.requires_grad_() for t in args)
    flat = x.reshape(B * S, d)
    logits = flat @ router_w
    probs = torch.softmax(logits, dim=-1)
    top, chosen = torch.topk(logits, k, dim=-1)
    gate = torch.softmax(top, dim=-1)
    out = torch.zeros((B * S, d), dtype=F64, device=DEVICE)
    load = torch.zeros(E, dtype=F64, device=DEVICE)
    for e in range(E):
        token, slot = torch.nonzero(chosen == e, as_tuple=True)
        load[e] = token.numel() / (B * S * k)
        mid = torch.nn.functional.gelu(flat[token] @ up_w[e] + up_b[e], approximate="tanh")
        out = out.index_add(0, token, (mid @ down_w[e] + down_b[e]) * gate[token, slot][:, None])
    mean_probability = probs.mean(0)
    summary = torch.stack((-(probs * torch.log(probs + 1.0e-9)).sum(-1).mean(), gate[:, 0].mean(),
                           logits.square().mean().sqrt())).detach()
    out = out.reshape(B, S, d)
    values = (out.detach(), mean_probability.detach(), load, summary)
    if not state["backward"]:
        return values
    return (*values, *torch.autograd.grad((out, mean_probability), (x, router_w, up_w, up_b, down_w, down_b),
                                          [t.to(F64) for t in state["douts"]]))
