"""GPU parity of the routed MLP (``gptrig.moe``) against the CPU oracle.

The oracle (``oracle/moe.py``) restates ``routed_mlp_local`` /
``load_balance_loss`` of ``recipes/reference_moe/train.py:1230-1371``.  Inputs
are drawn so that no token has two router logits within 1e-4 of each other
around the top-k boundary: the GPU's fp32 logits (a different summation
order) then route every token exactly as the oracle does, and the routing
indices are compared bit-exactly.  Tolerances: combined output and every
gradient max-abs <= 3e-2 of the reference's largest magnitude (bf16 chain of
two GEMMs, GELU and the bf16 scatter-add); mean probability <= 1e-5; load
exact; summary <= 1e-4 relative.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe as omoe

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def draw(batch, length, width, hidden, experts, seed):
    rng = np.random.default_rng(seed)

    def n(shape, std):
        return torch.from_numpy((rng.standard_normal(shape) * std).astype(np.float32))

    x = n((batch, length, width), 1.0).to(torch.bfloat16)
    router_w = n((width, experts), 0.1)
    up_w, up_b = n((experts, width, hidden), 0.05), n((experts, hidden), 0.05)
    down_w, down_b = n((experts, hidden, width), 0.05), n((experts, width), 0.05)
    return x, router_w, up_w, up_b, down_w, down_b


def routing_margin(x, router_w, top_k):
    logits = x.reshape(-1, x.shape[-1]).float() @ router_w
    srt = torch.sort(logits, dim=-1, descending=True).values
    return float((srt[:, : top_k] - srt[:, 1: top_k + 1]).min())


def maxabs(a, b):
    return float((a.detach().float().cpu() - b.detach().float().cpu()).abs().max())


def scale(t):
    return max(float(t.detach().float().abs().max()), 1e-6)


@pytest.mark.parametrize("batch,length,width,hidden,experts,top_k", [(4, 128, 256, 512, 8, 2), (2, 96, 128, 256, 4, 1),
                                                                     (2, 64, 128, 128, 6, 3)])
def test_routed_mlp_forward_backward_matches_oracle(batch, length, width, hidden, experts, top_k):
    from gptrig import moe

    print(f"moe case B={batch} L={length} D={width} F={hidden} E={experts} k={top_k}", flush=True)
    x, router_w, up_w, up_b, down_w, down_b = draw(batch, length, width, hidden, experts, 5)
    assert routing_margin(x, router_w, top_k) > 1e-4
    g = torch.from_numpy(np.random.default_rng(6).standard_normal((batch, length, width)).astype(np.float32))
    g = g.to(torch.bfloat16).float()
    aux = 0.01

    # Oracle: forward + autograd gradients.
    leaves = [t.clone().requires_grad_(True) for t in (x, router_w, up_w, up_b, down_w, down_b)]
    comb_r, mp_r, load_r, summ_r, chosen_r, gate_r = omoe.routed_mlp_local(
        *leaves, experts=experts, top_k_count=top_k, dtype=torch.bfloat16)
    loss_r = (comb_r.float() * g).sum() + aux * omoe.load_balance_loss(mp_r, load_r)
    grads_r = torch.autograd.grad(loss_r, leaves)

    # GPU.
    dev_leaves = [t.to(DEV).requires_grad_(True) for t in (x, router_w, up_w, up_b, down_w, down_b)]
    comb, mp, load, summ = moe.routed_mlp_local(*dev_leaves, experts=experts, top_k=top_k)
    loss = (comb.float() * g.to(DEV)).sum() + aux * moe.load_balance_loss(mp, load)
    grads = torch.autograd.grad(loss, dev_leaves)
    torch.cuda.synchronize()

    assert torch.equal(load.cpu(), load_r.detach())
    assert maxabs(mp, mp_r) <= 1e-5
    assert float(((summ.cpu() - summ_r.detach()).abs() / summ_r.detach().abs()).max()) <= 1e-4
    assert maxabs(comb, comb_r) <= 3e-2 * scale(comb_r)
    names = ("x", "router_w", "up_w", "up_b", "down_w", "down_b")
    for name, got, want in zip(names, grads, grads_r):
        err = maxabs(got, want)
        print(f"  d{name}: max-abs {err:.3e} (scale {scale(want):.3e})", flush=True)
        assert err <= 3e-2 * scale(want), name


def test_routing_indices_bit_exact_through_the_front_end():
    from gptrig import _lib
    from gptrig.moe import _route

    x, router_w, *_ = draw(2, 256, 256, 128, 8, 11)
    flat = x.reshape(-1, 256)
    logits_g, probs, chosen, gate, counts, rows, position = _route(flat.to(DEV).contiguous(), router_w.to(DEV), 8, 2)
    torch.cuda.synchronize()
    # Logits within fp32 summation-order noise; routing from the GPU's own logits bit-exact.
    logits_r = flat.float() @ router_w
    assert maxabs(logits_g, logits_r) <= 1e-5 * scale(logits_r) + 1e-6
    _, chosen_r, gate_r, order_r, _, counts_r, rows_r = omoe.route(logits_g.cpu(), 8, 2)
    assert torch.equal(chosen.cpu(), chosen_r)
    assert torch.equal(counts.cpu(), counts_r)
    assert torch.equal(rows.cpu().long(), rows_r)
    assert _lib.version()


def test_config_e_layer_shape_token_subset():
    """Config E's routed layer (32 x 1024 tokens, width 768, 8 experts of width
    3072, top-2) on the GPU; each token's output depends only on that token, so
    64 sampled tokens are checked against the oracle run on those tokens alone,
    and the input gradient of the same tokens likewise (no balance term)."""

    from gptrig import moe

    B, L, D, F, E, k = 32, 1024, 768, 3072, 8, 2
    rng = np.random.default_rng(21)

    def n(shape, std):
        return torch.from_numpy((rng.standard_normal(shape) * std).astype(np.float32))

    x = n((B, L, D), 1.0).to(torch.bfloat16)
    router_w = n((D, E), 0.02)
    up_w, up_b = n((E, D, F), 0.02), n((E, F), 0.02)
    down_w, down_b = n((E, F, D), 0.02), n((E, D), 0.02)
    g = n((B, L, D), 1.0).to(torch.bfloat16)
    xg = x.to(DEV).requires_grad_(True)
    params = [t.to(DEV) for t in (router_w, up_w, up_b, down_w, down_b)]
    comb, mp, load, summ = moe.routed_mlp_local(xg, *params, experts=E, top_k=k)
    (dx,) = torch.autograd.grad((comb.float() * g.to(DEV).float()).sum(), [xg])
    torch.cuda.synchronize()
    assert int(load.sum().mul(B * L * k).round()) == B * L * k
    flat_idx = torch.from_numpy(np.random.default_rng(22).choice(B * L, 64, replace=False))
    xs = x.reshape(B * L, D)[flat_idx].reshape(1, 64, D)
    assert routing_margin(xs, router_w, k) > 1e-5
    xs_leaf = xs.clone().requires_grad_(True)
    comb_r, *_ = omoe.routed_mlp_local(xs_leaf, router_w, up_w, up_b, down_w, down_b, experts=E, top_k_count=k,
                                       dtype=torch.bfloat16)
    gs = g.reshape(B * L, D)[flat_idx].reshape(1, 64, D).float()
    (dx_r,) = torch.autograd.grad((comb_r.float() * gs).sum(), [xs_leaf])
    got = comb.reshape(B * L, D)[flat_idx.to(DEV)]
    assert maxabs(got, comb_r.reshape(64, D)) <= 3e-2 * scale(comb_r)
    got_dx = dx.reshape(B * L, D)[flat_idx.to(DEV)]
    assert maxabs(got_dx, dx_r.reshape(64, D)) <= 3e-2 * scale(dx_r)


def test_config_e_routing_bit_exact_on_all_tokens():
    """Config E's routing at its full size (32 x 1024 = 32,768 tokens, width
    768, 8 experts, top-2, router ~ N(0, 0.02) as initialised): every token's
    expert indices, the per-expert counts, the stable bucket order (one
    1024-thread workgroup sorts all 65,536 assignments) and its inverse are
    bit-exact against the oracle's route of the GPU's own fp32 logits, the
    gates and probabilities within 1e-6.  A second pass plants integer logits
    (ties) in every 16th token to exercise the lower-index rule at this size."""
    from gptrig import _lib
    from gptrig.moe import _route

    T, D, E, k = 32 * 1024, 768, 8, 2
    rng = np.random.default_rng(2)
    x = torch.from_numpy(rng.standard_normal((T, D)).astype(np.float32)).to(torch.bfloat16)
    router_w = torch.from_numpy((rng.standard_normal((D, E)) * 0.02).astype(np.float32))
    print(f"config E routing, {T} tokens", flush=True)
    logits, probs, chosen, gate, counts, rows, position = _route(x.to(DEV), router_w.to(DEV), E, k)
    torch.cuda.synchronize()
    probs_r, chosen_r, gate_r, order_r, _, counts_r, rows_r = omoe.route(logits.cpu(), E, k)
    assert torch.equal(chosen.cpu(), chosen_r)
    assert torch.equal(counts.cpu(), counts_r)
    assert torch.equal(rows.cpu().long(), rows_r)
    inv = torch.empty_like(order_r)
    inv[order_r] = torch.arange(T * k)
    assert torch.equal(position.cpu().long(), inv)
    assert maxabs(gate, gate_r) <= 1e-6 and maxabs(probs, probs_r) <= 1e-6

    tied = logits.cpu().clone()
    tied[::16] = torch.from_numpy(rng.integers(-2, 3, size=(T // 16, E)).astype(np.float32))
    probs_r, chosen_r, gate_r, order_r, _, counts_r, rows_r = omoe.route(tied, E, k)
    lg = tied.to(DEV)
    order = torch.empty(T * k, dtype=torch.int32, device=DEV)
    ws = _lib.workspace(_lib.query("gptrig_moe_route_workspace_bytes", T, E, k), lg.device)
    _lib.call("gptrig_moe_route", lg.data_ptr(), probs.data_ptr(), chosen.data_ptr(), gate.data_ptr(),
              counts.data_ptr(), order.data_ptr(), rows.data_ptr(), position.data_ptr(), ws.data_ptr(), ws.numel(),
              T, E, k, _lib.stream())
    torch.cuda.synchronize()
    assert torch.equal(chosen.cpu(), chosen_r)
    assert torch.equal(counts.cpu(), counts_r)
    assert torch.equal(order.cpu().long(), order_r)
    assert torch.equal(rows.cpu().long(), rows_r)


@pytest.mark.parametrize("tokens,width,experts", [
    (1, 8, 1), (15, 40, 3), (64, 256, 16), (65, 520, 8), (200, 96, 5), (33, 36, 4),  # (33, 36): element loads
])
def test_router_logits_against_float64(tokens, width, experts):
    """The split-weight router product at its edges (one token, ragged token
    tiles, widths with partial steps and without 16-byte loads, every expert
    count class) against float64.

    Bound: exact products, three float32 sums of ``width`` of them rounded
    once per 32 and added: 2^-24 (ceil(width / 32) + 3) of the magnitudes."""
    from gptrig import _lib

    g = torch.Generator().manual_seed(width)
    x = torch.randn((tokens, width), generator=g).bfloat16().to(DEV)
    w = (torch.randn((width, experts), generator=g) * 0.3).to(DEV)
    logits = torch.full((tokens, experts), float("nan"), device=DEV)
    print(f"router logits tokens={tokens} width={width} experts={experts}", flush=True)
    _lib.call("gptrig_moe_router_logits", x.data_ptr(), w.data_ptr(), logits.data_ptr(), tokens, width, experts,
              _lib.stream())
    x64, w64 = x.double(), w.double()
    bound = (x64.abs() @ w64.abs()) * 2.0 ** -24 * (-(-width // 32) + 3)
    excess = float(((logits.double() - x64 @ w64).abs() / bound).max())
    print(f"  error / bound {excess:.3f}", flush=True)
    assert excess <= 1


@pytest.mark.parametrize("tokens,width,experts", [(70, 64, 8), (17, 36, 3)])
def test_router_logits_of_infinite_operands(tokens, width, experts):
    """Infinite weights, activations and products give the infinities and NaN
    of a float32 sum of products, in their own tokens and experts alone."""
    from gptrig import _lib

    g = torch.Generator().manual_seed(tokens)
    x = torch.rand((tokens, width), generator=g).add(0.1).bfloat16().to(DEV)
    w = (torch.randn((width, experts), generator=g) * 0.3).to(DEV)
    logits = torch.empty((tokens, experts), device=DEV)
    run = lambda: _lib.call("gptrig_moe_router_logits", x.data_ptr(), w.data_ptr(), logits.data_ptr(), tokens,  # noqa: E731
                            width, experts, _lib.stream())
    print(f"router infinities tokens={tokens} width={width} experts={experts}", flush=True)
    run()
    before = logits.clone()
    w[3, 0] = -torch.inf
    w[5, 1] = torch.inf
    x[4, 7] = torch.inf
    x[6, 2] = torch.nan
    run()
    sign = torch.sign(w[7].double())
    want = before.clone()
    want[:, 0], want[:, 1] = -torch.inf, torch.inf
    for e in range(experts):
        inf = float(sign[e]) * torch.inf
        want[4, e] = inf if e > 1 or want[4, e] == inf else torch.nan
    want[6] = torch.nan
    assert torch.equal(torch.nan_to_num(logits, 7e37, 8e37, -9e37), torch.nan_to_num(want, 7e37, 8e37, -9e37))


@pytest.mark.parametrize("tokens,width,experts,top_k", [
    (1, 8, 2, 1), (255, 64, 4, 2), (257, 72, 8, 2), (300, 136, 16, 3), (130, 264, 5, 1),
    (2048, 4096, 2, 2), (2047, 4096, 2, 1),  # two workgroups per CU (of 256) or just not: runs of one and two tiles
])
def test_fused_input_backward_equals_two_passes(tokens, width, experts, top_k):
    """gptrig_moe_input_bwd against gptrig_moe_gather_bwd then
    gptrig_moe_router_bwd: dx bit for bit, the router gradient to its float32
    atomics (each workgroup adds one partial per entry)."""
    from gptrig import _lib

    g = torch.Generator().manual_seed(tokens + width)
    R = tokens * top_k
    x, dgrouped = (torch.randn((n, width), generator=g).bfloat16().to(DEV) for n in (tokens, R))
    w = (torch.randn((width, experts), generator=g) * 0.1).to(DEV)
    probs = torch.softmax(torch.randn((tokens, experts), generator=g), -1).to(DEV)
    chosen = torch.rand((tokens, experts), generator=g).topk(top_k).indices.to(torch.int32).to(DEV)
    gate = torch.softmax(torch.randn((tokens, top_k), generator=g), -1).to(DEV)
    dgate, dmean = torch.randn(R, generator=g).to(DEV), torch.randn(experts, generator=g).to(DEV)
    position = torch.randperm(R, generator=g).to(torch.int32).to(DEV)
    s = _lib.stream()
    print(f"input backward tokens={tokens} width={width} experts={experts} top_k={top_k}", flush=True)
    tail = [probs, chosen, gate, dgate, dmean]
    dx1, dx2 = (torch.full((tokens, width), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    dw1, dw2 = (torch.ones((width, experts), device=DEV) for _ in range(2))
    _lib.call("gptrig_moe_gather_bwd", dgrouped.data_ptr(), position.data_ptr(), dx1.data_ptr(), tokens, width, top_k, s)
    _lib.call("gptrig_moe_router_bwd", x.data_ptr(), w.data_ptr(), *(t.data_ptr() for t in tail), dx1.data_ptr(),
              dw1.data_ptr(), tokens, width, experts, top_k, s)
    _lib.call("gptrig_moe_input_bwd", dgrouped.data_ptr(), position.data_ptr(), x.data_ptr(), w.data_ptr(),
              *(t.data_ptr() for t in tail), dx2.data_ptr(), dw2.data_ptr(), tokens, width, experts, top_k, s)
    assert torch.equal(dx1, dx2)
    torch.testing.assert_close(dw1, dw2, rtol=1e-6, atol=1e-5 * float(dw1.abs().max()))


@pytest.mark.parametrize("counts,width,hidden", [
    ([5], 8, 16),                        # one expert, a corner of a tile
    ([0, 33, 0, 7], 264, 72),            # empty experts (their gradients are zero), ragged tiles
    ([3000, 10, 0, 200], 64, 520),       # one expert far over the even share: sliced, added with atomics
    ([700, 650, 720, 690, 10, 1, 0, 629], 256, 256),
])
def test_backward_gemms_in_one_launch(counts, width, hidden):
    """gptrig_moe_bwd_gemms against float64 for every kind of bucket: stored,
    sliced and empty ones; the outputs start as NaN.

    Bound: bf16 products are exact in float32 and a sum of n rounds at most n
    times, 2^-24 n of the magnitudes; dgrouped is rounded to bf16 once."""
    from gptrig import _lib

    g = torch.Generator().manual_seed(width + hidden)
    E, R = len(counts), sum(counts)
    rnd = lambda *s: torch.randn(s, generator=g).bfloat16().to(DEV)  # noqa: E731
    grouped, dpre, hid, dout, up_w = rnd(R, width), rnd(R, hidden), rnd(R, hidden), rnd(R, width), rnd(E, width, hidden)
    cnt = torch.tensor(counts, dtype=torch.int32, device=DEV)
    nan = lambda *s, dtype=torch.float32: torch.full(s, float("nan"), dtype=dtype, device=DEV)  # noqa: E731
    up_dw, up_db, down_dw, down_db = nan(E, width, hidden), nan(E, hidden), nan(E, hidden, width), nan(E, width)
    dgrouped = nan(R, width, dtype=torch.bfloat16)
    print(f"routed backward products counts={counts} width={width} hidden={hidden}", flush=True)
    _lib.call("gptrig_moe_bwd_gemms", grouped.data_ptr(), dpre.data_ptr(), hid.data_ptr(), dout.data_ptr(),
              up_w.data_ptr(), cnt.data_ptr(), up_dw.data_ptr(), up_db.data_ptr(), down_dw.data_ptr(),
              down_db.data_ptr(), dgrouped.data_ptr(), R, width, hidden, E, _lib.stream())
    worst, at = 0.0, 0
    for e, n in enumerate(counts):
        a, p, h, o = (t[at:at + n].double() for t in (grouped, dpre, hid, dout))
        eps = (n + 2) * 2.0 ** -24
        for got, x, y in ((up_dw[e], a, p), (down_dw[e], h, o)):
            bound = eps * (x.abs().T @ y.abs()) + 1e-30
            worst = max(worst, float(((got.double() - x.T @ y).abs() / bound).max()))
        for got, y in ((up_db[e], p), (down_db[e], o)):
            worst = max(worst, float(((got.double() - y.sum(0)).abs() / (eps * y.abs().sum(0) + 1e-30)).max()))
        w = up_w[e].double()
        want = p @ w.T
        bound = (hidden + 2) * 2.0 ** -24 * (p.abs() @ w.abs().T) + 2.0 ** -8 * want.abs() + 1e-30
        if n:
            worst = max(worst, float(((dgrouped[at:at + n].double() - want).abs() / bound).max()))
        at += n
    print(f"  error / bound {worst:.3f}", flush=True)
    assert worst <= 1


@pytest.mark.parametrize("dtypes,offset", [("ffff", 0), ("fbfb", 0), ("ffff", 1), ("bbbb", 0), ("hfff", 0)])
def test_routed_weights_of_any_dtype_and_base(dtypes, offset):
    """The weight casts in front of the routed MLP: float32 parameters
    (16-byte aligned or not, sizes with a tail of 8), bf16 and half ones give
    the layer the same bf16 operands as .to(bfloat16), and gradients come back in
    each parameter's dtype."""
    from gptrig import _lib
    from gptrig.moe import _bf16, routed_mlp_local

    kinds = {"f": torch.float32, "b": torch.bfloat16, "h": torch.float16}
    x, router_w, *params = draw(1, 9, 24, 40, 3, 3)
    on = []
    for t, k in zip(params, dtypes):
        flat = torch.zeros(t.numel() + offset, dtype=kinds[k], device=DEV)
        flat[offset:] = t.reshape(-1).to(kinds[k]).to(DEV)
        on.append(flat[offset:].view(t.shape))
    print(f"routed weights {dtypes} base {[t.data_ptr() % 16 for t in on]}", flush=True)
    for got, t in zip(_bf16(*on), on):
        assert got.is_contiguous() and torch.equal(got, t.to(torch.bfloat16))
    leaves = [t.detach().requires_grad_() for t in on]
    out, *_ = routed_mlp_local(x.to(DEV), router_w.to(DEV), *leaves, experts=3, top_k=2)
    grads = torch.autograd.grad(out.float().sum(), leaves)
    assert all(g.dtype == t.dtype and g.shape == t.shape and torch.isfinite(g).all() for g, t in zip(grads, leaves))
    same = [t.detach().to(torch.bfloat16).requires_grad_() for t in on]
    ref, *_ = routed_mlp_local(x.to(DEV), router_w.to(DEV), *same, experts=3, top_k=2)
    assert torch.equal(out, ref)
    saved = _lib.query("gptrig_routed_saved_bytes", 9, 24, 40, 3, 2)
    assert saved > 0 and _lib.query("gptrig_routed_saved_bytes", 0, 24, 40, 3, 2) == 0
