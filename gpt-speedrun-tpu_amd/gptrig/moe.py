"""Top-k routed MLP on the gfx950 kernels.

Mirrors ``routed_mlp_local`` and ``load_balance_loss`` of
``recipes/reference_moe/train.py:1230-1307,1347-1371`` on one device (the
``axis_name`` reductions collapse): fp32 router logits, ``jax.lax.top_k``
routing with a stable bucket sort, two grouped expert GEMMs (``megablox.gmm``)
with bias / GELU epilogues, and the gated scatter-add.  Forward and backward
run entirely in ``libgptrig.so``; torch only allocates.
"""

from __future__ import annotations

import ctypes

import torch

from . import _lib

BF16 = torch.bfloat16
F32 = torch.float32


def _route(flat: torch.Tensor, router_w: torch.Tensor, experts: int, top_k: int, ws: torch.Tensor | None = None):
    """Router logits and bucket routing of the bf16 rows ``flat`` alone (the
    trainer's routed block); ``ws``: a workspace to reuse."""

    tokens, width = flat.shape
    dev = flat.device
    s = _lib.stream()
    logits = torch.empty((tokens, experts), dtype=F32, device=dev)
    _lib.call("gptrig_moe_router_logits", flat.data_ptr(), router_w.data_ptr(), logits.data_ptr(), tokens, width,
              experts, s)
    probs = torch.empty((tokens, experts), dtype=F32, device=dev)
    chosen = torch.empty((tokens, top_k), dtype=torch.int32, device=dev)
    gate = torch.empty((tokens, top_k), dtype=F32, device=dev)
    counts = torch.empty(experts, dtype=torch.int32, device=dev)
    order = torch.empty(tokens * top_k, dtype=torch.int32, device=dev)
    rows = torch.empty(tokens * top_k, dtype=torch.int32, device=dev)
    position = torch.empty(tokens * top_k, dtype=torch.int32, device=dev)
    if ws is None:
        ws = _lib.workspace(_lib.query("gptrig_moe_route_workspace_bytes", tokens, experts, top_k), dev)
    _lib.call("gptrig_moe_route", logits.data_ptr(), probs.data_ptr(), chosen.data_ptr(), gate.data_ptr(),
              counts.data_ptr(), order.data_ptr(), rows.data_ptr(), position.data_ptr(), ws.data_ptr(), ws.numel(),
              tokens, experts, top_k, s)
    return logits, probs, chosen, gate, counts, rows, position


def _bf16(*tensors: torch.Tensor) -> list[torch.Tensor]:
    """Contiguous bf16 copies (float32 tensors in one launch); bf16 ones as they are."""

    out = [t if t.dtype == F32 else t.to(BF16).contiguous() for t in tensors]
    todo = [i for i, t in enumerate(out) if t.dtype == F32]
    if not todo:
        return out
    src = [out[i].contiguous() for i in todo]
    src = [t.clone() if t.data_ptr() % 16 else t for t in src]  # (a view into an arena at an odd element)
    dst = [torch.empty(t.shape, dtype=BF16, device=t.device) for t in src]
    n = len(src)
    _lib.call("gptrig_cast_f32_bf16_many", (ctypes.c_void_p * n)(*(t.data_ptr() for t in src)),
              (ctypes.c_void_p * n)(*(t.data_ptr() for t in dst)), (ctypes.c_int64 * n)(*(t.numel() for t in src)), n,
              _lib.stream())
    for i, t in zip(todo, dst):
        out[i] = t
    return out


class _RoutedMLP(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, router_w, up_w, up_b, down_w, down_b, experts: int, top_k: int):
        batch, length, width = x.shape
        tokens = batch * length
        hidden_width = up_w.shape[-1]
        dev = x.device
        flat = x.reshape(tokens, width).to(BF16).contiguous()
        rw = router_w.to(F32).contiguous()
        upw, upb, dnw, dnb = _bf16(up_w, up_b, down_w, down_b)
        sizes = (tokens, width, hidden_width, experts, top_k)
        saved = _lib.workspace(_lib.query("gptrig_routed_saved_bytes", *sizes), dev)
        scratch = _lib.workspace(_lib.query("gptrig_routed_scratch_bytes", *sizes, 0), dev)
        combined = torch.empty((tokens, width), dtype=BF16, device=dev)
        mean_probability = torch.empty(experts, dtype=F32, device=dev)
        load = torch.empty(experts, dtype=F32, device=dev)
        summary = torch.empty(3, dtype=F32, device=dev)
        _lib.call("gptrig_routed_fwd", flat.data_ptr(), rw.data_ptr(), upw.data_ptr(), upb.data_ptr(), dnw.data_ptr(),
                  dnb.data_ptr(), combined.data_ptr(), mean_probability.data_ptr(), load.data_ptr(),
                  summary.data_ptr(), saved.data_ptr(), saved.numel(), scratch.data_ptr(), scratch.numel(), *sizes,
                  _lib.stream())
        ctx.save_for_backward(flat, rw, upw, dnw, saved)
        ctx.meta = (batch, length, sizes, x.dtype, router_w.dtype, up_w.dtype, up_b.dtype, down_w.dtype, down_b.dtype)
        ctx.mark_non_differentiable(load, summary)
        return combined.reshape(batch, length, width).to(x.dtype), mean_probability, load, summary

    @staticmethod
    def backward(ctx, dcombined, dmean_probability, _dload, _dsummary):
        flat, rw, upw, dnw, saved = ctx.saved_tensors
        batch, length, sizes, xdt, rdt, uwdt, ubdt, dwdt, dbdt = ctx.meta
        tokens, width, hidden_width, experts, top_k = sizes
        dev = flat.device
        if dcombined is None:
            dcombined = torch.zeros((tokens, width), dtype=BF16, device=dev)
        dc = dcombined.reshape(tokens, width).to(BF16).contiguous()
        dmp = None if dmean_probability is None else dmean_probability.to(F32).contiguous()
        dx = torch.empty((tokens, width), dtype=BF16, device=dev)
        d_up_w = torch.empty((experts, width, hidden_width), dtype=F32, device=dev)
        d_up_b = torch.empty((experts, hidden_width), dtype=F32, device=dev)
        d_down_w = torch.empty((experts, hidden_width, width), dtype=F32, device=dev)
        d_down_b = torch.empty((experts, width), dtype=F32, device=dev)
        d_router = torch.empty((width, experts), dtype=F32, device=dev)
        scratch = _lib.workspace(_lib.query("gptrig_routed_scratch_bytes", *sizes, 1), dev)
        _lib.call("gptrig_routed_bwd", dc.data_ptr(), _lib.ptr(dmp), flat.data_ptr(), rw.data_ptr(), upw.data_ptr(),
                  dnw.data_ptr(), saved.data_ptr(), saved.numel(), dx.data_ptr(), d_router.data_ptr(),
                  d_up_w.data_ptr(), d_up_b.data_ptr(), d_down_w.data_ptr(), d_down_b.data_ptr(), scratch.data_ptr(),
                  scratch.numel(), *sizes, _lib.stream())
        return (dx.reshape(batch, length, width).to(xdt), d_router.to(rdt), d_up_w.to(uwdt), d_up_b.to(ubdt),
                d_down_w.to(dwdt), d_down_b.to(dbdt), None, None)


def routed_mlp_local(x: torch.Tensor, router_w: torch.Tensor, up_w: torch.Tensor, up_b: torch.Tensor,
                     down_w: torch.Tensor, down_b: torch.Tensor, *, experts: int, top_k: int,
                     dtype=torch.bfloat16, axis_name=None):
    """``routed_mlp_local`` (``reference_moe/train.py:1230-1307``) on one device.

    ``x`` [batch, length, width]; ``router_w`` [width, experts] (fp32 math);
    ``up_w`` [experts, width, hidden], ``up_b`` [experts, hidden], ``down_w``
    [experts, hidden, width], ``down_b`` [experts, width].  Returns
    ``(combined, mean_probability, load, summary)``; ``load`` and ``summary``
    carry no gradient (``load`` is a count ratio, as in the reference).
    """

    if dtype != torch.bfloat16:
        raise TypeError("the routed MLP kernels compute in bfloat16")
    if axis_name is not None:
        raise ValueError("one device: the data-axis reductions collapse; pass axis_name=None")
    if x.ndim != 3:
        raise ValueError(f"x must be [batch, length, width], got {tuple(x.shape)}")
    width = x.shape[-1]
    hidden = up_w.shape[-1]
    if router_w.shape != (width, experts):
        raise ValueError(f"router_w must be [{width}, {experts}], got {tuple(router_w.shape)}")
    if up_w.shape != (experts, width, hidden) or up_b.shape != (experts, hidden):
        raise ValueError("up_w / up_b must be [experts, width, hidden] / [experts, hidden]")
    if down_w.shape != (experts, hidden, width) or down_b.shape != (experts, width):
        raise ValueError("down_w / down_b must be [experts, hidden, width] / [experts, width]")
    if not 0 < top_k <= experts:
        raise ValueError(f"top_k must be in [1, experts], got {top_k}")
    _lib.require_device(x, router_w, up_w, up_b, down_w, down_b)
    return _RoutedMLP.apply(x, router_w, up_w, up_b, down_w, down_b, int(experts), int(top_k))


def load_balance_loss(mean_probability: torch.Tensor, load: torch.Tensor) -> torch.Tensor:
    """``load_balance_loss`` (``reference_moe/train.py:1347-1371``): ``E * sum(load * P)``."""

    if mean_probability.ndim != 1 or load.ndim != 1:
        raise ValueError("load_balance_loss takes per-expert vectors already reduced over tokens, got shapes "
                         f"{tuple(mean_probability.shape)} and {tuple(load.shape)}")
    return float(load.shape[0]) * (load * mean_probability).sum()
