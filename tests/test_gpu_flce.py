"""GPU parity of the FLCE backward's paths, through the C ABI (ctypes).

* the chunked backward (several vocabulary chunks: the public API's default
  ``vocab_tile_size`` = 2048, pipelined launches over two halves of the
  ``[tokens, chunk]`` buffer), the one-chunk launches and the kept-softmax
  pair (the trainer's whole-vocabulary opt-in: the forward keeps its fp16
  probabilities, the backward rescales them instead of recomputing the
  logits) against the CPU oracle (``oracle.flce``, restating
  ``rig/kernels/linear_cross_entropy.py``), at config C's full size (16384
  tokens x 768 x 50304) and at small ragged shapes;
* the reference's width-5 bfloat16 fixture (``tests/test_linear_cross_entropy.py:
  73-80,129-152``), through the zero-padded public API.

Tolerances: mean loss relative error <= 1e-3 (north star), per-token loss
``1e-3 |loss| + 2e-4``, dh and dW max-abs <= 2% of their largest magnitude
(bf16 operands of the reference's own tiled matmuls).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import flce as oflce

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def maxabs(a, b):
    return float((a.float().cpu() - b.float().cpu()).abs().max())


def inputs(n, d, V, sv, seed, h_scale=1.0, w_scale=0.02):
    g = torch.Generator().manual_seed(seed)
    h = (torch.randn((n, d), generator=g) * h_scale).to(torch.bfloat16)
    w = torch.randn((V, d), generator=g) * w_scale
    t = torch.randint(0, sv, (n,), generator=g, dtype=torch.int32)
    return h, w, t


def run_backward(h, w, t, sv, chunk, ct=None, scale=0.0, dweight=None, accumulate=False):
    from gptrig.kernels import linear_cross_entropy as lce

    hg, wg, tg = h.to(DEV), w.to(torch.bfloat16).to(DEV), t.to(DEV)
    losses, lse = lce.flce_forward(hg, wg, tg, sv)
    dh, dw = lce.flce_backward(hg, wg, tg, lse, None if ct is None else ct.to(DEV), scale, sv, chunk,
                               dweight=dweight, accumulate=accumulate)
    torch.cuda.synchronize()
    return losses.cpu(), lse.cpu(), dh.cpu(), dw.cpu()


@pytest.mark.skip(reason="ran the in-kernel work-queue FLCE backward (cross-workgroup dependency counters), which "
                         "went silent for 180 s on its first GPU run with no cause found by reading; that kernel is "
                         "removed, and the chunked path (pipelined launches, no waits inside a launch) is covered by "
                         "test_config_c_pipelined_default_tile_matches_oracle")
def test_config_c_default_tile_and_whole_vocabulary_match_oracle():
    """Config C (16384 x 768 x 50304) through the removed work-queue kernel."""


def test_config_c_pipelined_default_tile_matches_oracle():
    """Config C (16384 x 768 x 50304, W ~ N(0, 0.02), mean loss): the public
    API's default tile (2048: 50 chunks of 1024 rows, 51 pipelined launches)
    and the trainer's single chunk against the oracle's tiled reference."""
    import time

    from gptrig.kernels import linear_cross_entropy as lce

    n, d, V = 16384, 768, 50304
    print(f"flce config C n={n} d={d} V={V}: oracle on the CPU", flush=True)
    h, w, t = inputs(n, d, V, V, 51)
    torch.set_num_threads(16)
    t0 = time.time()
    losses_ref, lse_ref = oflce.losses_and_lse(h, w, t, semantic_vocab_size=V, vocab_tile_size=2048)
    print(f"oracle forward {time.time() - t0:.1f} s", flush=True)
    ct = torch.full((n,), 1.0 / n)
    dh_ref, dw_ref = oflce.losses_backward(h, w, t, lse_ref, ct, semantic_vocab_size=V, vocab_tile_size=2048)
    print(f"oracle backward done {time.time() - t0:.1f} s; GPU public API", flush=True)
    sh, sw = float(dh_ref.float().abs().max()), float(dw_ref.abs().max())
    # Public API, default vocab_tile_size (2048).
    hg = h.to(DEV).requires_grad_(True)
    wg = w.to(DEV).requires_grad_(True)
    loss = lce.tiled_tied_cross_entropy(hg, wg, t.to(DEV), semantic_vocab_size=V)
    loss.backward()
    torch.cuda.synchronize()
    want = float(losses_ref.mean())
    print(f"mean loss gpu {float(loss):.6f} oracle {want:.6f}; dh {maxabs(hg.grad, dh_ref) / sh:.4f}, "
          f"dW {maxabs(wg.grad, dw_ref) / sw:.4f} of max", flush=True)
    assert abs(float(loss) - want) <= 1e-3 * abs(want)
    assert maxabs(hg.grad, dh_ref) <= 2e-2 * sh
    assert maxabs(wg.grad, dw_ref) <= 2e-2 * sw
    # Trainer opt-in: one chunk, scalar cotangent.
    print("GPU one chunk", flush=True)
    _, _, dh1, dw1 = run_backward(h, w, t, V, lce.grad_chunk(n, V), scale=1.0 / n)
    assert maxabs(dh1, dh_ref) <= 2e-2 * sh
    assert maxabs(dw1, dw_ref) <= 2e-2 * sw
    # The two paths sum the same bf16 products in different fp32 orders.
    assert maxabs(dh1, hg.grad) <= 1e-2 * sh
    # Kept-softmax pair (the trainer's path): same losses as the forward, and
    # gradients from the rescaled kept probabilities.
    print("GPU kept softmax", flush=True)
    lk, lsek, dhk, dwk = run_keep(h, w, t, V, scale=1.0 / n)
    assert abs(float(lk.mean()) - want) <= 1e-3 * abs(want)
    assert maxabs(dhk, dh_ref) <= 2e-2 * sh
    assert maxabs(dwk, dw_ref) <= 2e-2 * sw
    assert maxabs(dhk, dh1) <= 1e-2 * sh and maxabs(dwk, dw1) <= 1e-2 * sw


def run_keep(h, w, t, sv, ct=None, scale=0.0, dweight=None, accumulate=False):
    from gptrig.kernels import linear_cross_entropy as lce

    hg, wg, tg = h.to(DEV), w.to(torch.bfloat16).to(DEV), t.to(DEV)
    losses, lse, keep = lce.flce_forward_keep(hg, wg, tg, sv)
    dh, dw = lce.flce_backward_keep(hg, wg, tg, lse, keep, None if ct is None else ct.to(DEV), scale, sv,
                                    dweight=dweight, accumulate=accumulate)
    torch.cuda.synchronize()
    return losses.cpu(), lse.cpu(), dh.cpu(), dw.cpu()


KEEP_CASES = [
    # (n, d, V, semantic V): ragged vocabulary tiles and a partial last token tile; d a multiple of 128
    (2056, 256, 1300, 1297),
    (4096, 768, 5000, 4999),
    (8, 128, 600, 600),
    (1536, 384, 2312, 2000),
]


@pytest.mark.parametrize("n,d,V,sv", KEEP_CASES)
def test_kept_softmax_pair_matches_oracle_and_forward(n, d, V, sv):
    """gptrig_flce_fwd_keep / gptrig_flce_bwd_keep: the forward's losses and
    lse equal gptrig_flce_fwd's bit for bit (same launches plus stores), and
    the gradients from the rescaled kept probabilities match the oracle to the
    tolerances of the recompute path (one more fp16 rounding per probability),
    with invalid targets, per-token cotangents, padding rows and dW
    accumulation."""
    print(f"flce kept case n={n} d={d} V={V} sv={sv}", flush=True)
    h, w, t = inputs(n, d, V, sv, 71, 0.5, 0.5)
    t[::11] = -1
    g = torch.Generator().manual_seed(72)
    ct = torch.rand(n, generator=g)
    losses_ref, lse_ref = oflce.losses_and_lse(h, w, t, semantic_vocab_size=sv, vocab_tile_size=256)
    dh_ref, dw_ref = oflce.losses_backward(h, w, t, lse_ref, ct, semantic_vocab_size=sv, vocab_tile_size=256)
    lo, ls, _, _ = run_backward(h, w, t, sv, 1 << 20, ct=ct)
    lk, lsk, dhk, dwk = run_keep(h, w, t, sv, ct=ct)
    assert torch.equal(torch.isfinite(lk), torch.isfinite(lo))
    fin = torch.isfinite(lo)
    assert torch.equal(lk[fin], lo[fin]) and torch.equal(lsk, ls)
    sh, sw = float(dh_ref.float().abs().max()), float(dw_ref.abs().max())
    print(f"  dh {maxabs(dhk, dh_ref) / sh:.4f}, dW {maxabs(dwk, dw_ref) / sw:.4f} of max", flush=True)
    assert maxabs(dhk, dh_ref) <= 2e-2 * sh
    assert maxabs(dwk, dw_ref) <= 2e-2 * sw
    assert (dwk[sv:] == 0).all()
    base = torch.randn(V, d, generator=g)
    _, _, dh2, dw2 = run_keep(h, w, t, sv, ct=ct, dweight=base.to(DEV), accumulate=True)
    # (The one-chunk dh GEMM adds its K splits with f32 atomics: equal up to
    # the order of those adds, one bf16 step at most.)
    assert maxabs(dh2, dhk) <= 1e-2 * sh
    assert maxabs(dw2 - base, dwk) <= 1e-5 * max(1.0, float(base.abs().max()))


def test_kept_softmax_token_chunks_equal_one_chunk():
    """The trainer's bounded form of the kept-softmax pair: the tokens cut into
    chunks (of 1024 and a ragged 520), each chunk's forward and backward run
    back to back with dW accumulated, against the oracle and against one call
    over all tokens.  Losses and lse are per token, so they are bit-equal; dh
    rows are per token too (equal up to the dh GEMM's split-K order); dW sums
    the chunks in another order (f32)."""
    from gptrig.kernels import linear_cross_entropy as lce

    n, d, V, sv = 3592, 256, 3000, 2998
    print(f"flce kept token chunks n={n} d={d} V={V}", flush=True)
    h, w, t = inputs(n, d, V, sv, 81, 0.5, 0.5)
    t[::13] = -1
    losses_ref, lse_ref = oflce.losses_and_lse(h, w, t, semantic_vocab_size=sv, vocab_tile_size=256)
    ct = torch.full((n,), 1.0 / n)
    dh_ref, dw_ref = oflce.losses_backward(h, w, t, lse_ref, ct, semantic_vocab_size=sv, vocab_tile_size=256)
    l1, ls1, dh1, dw1 = run_keep(h, w, t, sv, scale=1.0 / n)
    hg, wg, tg = h.to(DEV), w.to(torch.bfloat16).to(DEV), t.to(DEV)
    dw = torch.empty(V, d, device=DEV)
    parts_l, parts_s, parts_dh = [], [], []
    keep = None
    for c0 in range(0, n, 1024):
        c1 = min(n, c0 + 1024)
        lc, lsc, keep = lce.flce_forward_keep(hg[c0:c1], wg, tg[c0:c1], sv, keep)
        dhc, _ = lce.flce_backward_keep(hg[c0:c1], wg, tg[c0:c1], lsc, keep, None, 1.0 / n, sv, dweight=dw,
                                        accumulate=c0 > 0)
        parts_l.append(lc.cpu())
        parts_s.append(lsc.cpu())
        parts_dh.append(dhc.cpu())
    torch.cuda.synchronize()
    lk, lsk, dhk, dwk = torch.cat(parts_l), torch.cat(parts_s), torch.cat(parts_dh), dw.cpu()
    fin = torch.isfinite(l1)
    assert torch.equal(torch.isfinite(lk), fin) and torch.equal(lk[fin], l1[fin]) and torch.equal(lsk, ls1)
    sh, sw = float(dh_ref.float().abs().max()), float(dw_ref.abs().max())
    print(f"  dh {maxabs(dhk, dh_ref) / sh:.4f}, dW {maxabs(dwk, dw_ref) / sw:.4f} of max", flush=True)
    assert maxabs(dhk, dh_ref) <= 2e-2 * sh and maxabs(dwk, dw_ref) <= 2e-2 * sw
    assert maxabs(dhk, dh1) <= 1e-2 * sh
    assert maxabs(dwk, dw1) <= 1e-3 * sw
    assert (dwk[sv:] == 0).all()


CHUNKED_CASES = [
    # (n, d, V, semantic V, chunk): ragged token tiles, partial d tiles, ragged last chunks, the
    # alternating (256-row chunk) and pipelined (>= 512) forms
    (2056, 192, 1300, 1297, 512),
    (4096, 768, 5000, 4999, 1024),
    (8, 64, 600, 600, 256),
    (1536, 320, 2311, 2000, 768),
    (296, 128, 1000, 997, 256),
]


@pytest.mark.parametrize("n,d,V,sv,chunk", CHUNKED_CASES)
def test_chunked_backward_matches_oracle(n, d, V, sv, chunk):
    print(f"flce chunked case n={n} d={d} V={V} sv={sv} chunk={chunk}", flush=True)
    h, w, t = inputs(n, d, V, sv, 61, 0.5, 0.5)
    t[::13] = -1  # invalid targets: no gradient
    g = torch.Generator().manual_seed(62)
    ct = torch.rand(n, generator=g)
    losses_ref, lse_ref = oflce.losses_and_lse(h, w, t, semantic_vocab_size=sv, vocab_tile_size=chunk)
    dh_ref, dw_ref = oflce.losses_backward(h, w, t, lse_ref, ct, semantic_vocab_size=sv, vocab_tile_size=chunk)
    losses, lse, dh, dw = run_backward(h, w, t, sv, chunk, ct=ct)
    finite = torch.isfinite(losses_ref)
    assert torch.equal(finite, torch.isfinite(losses))
    assert bool(((losses[finite] - losses_ref[finite]).abs() <= 1e-3 * losses_ref[finite].abs() + 2e-4).all())
    sh, sw = float(dh_ref.float().abs().max()), float(dw_ref.abs().max())
    assert maxabs(dh, dh_ref) <= 2e-2 * sh
    assert maxabs(dw, dw_ref) <= 2e-2 * sw
    assert (dw[sv:] == 0).all()
    # accumulate_dweight: adds into an existing dW; the second call sees the same inputs.
    base = torch.randn(V, d, generator=g)
    _, _, dh2, dw2 = run_backward(h, w, t, sv, chunk, ct=ct, dweight=base.to(DEV), accumulate=True)
    assert torch.equal(dh2, dh)
    assert maxabs(dw2 - base, dw) <= 1e-5 * max(1.0, float(base.abs().max()))


def test_width_five_bfloat16_fixture():
    """tests/test_linear_cross_entropy.py:129-152 of the reference: hidden
    (2, 3, 5) from default_rng(7) as bfloat16, embedding (13, 5) from
    default_rng(11), semantic vocabulary 11, tile 7; the value within
    4e-3 of the dense bf16 oracle, gradients in the input dtypes."""
    from gptrig.kernels import tiled_tied_cross_entropy

    hidden = torch.from_numpy(np.random.default_rng(7).normal(size=(2, 3, 5)).astype(np.float32)).to(torch.bfloat16)
    embedding = torch.from_numpy(np.random.default_rng(11).normal(size=(13, 5)).astype(np.float32))
    targets = torch.tensor([[0, 1, 10], [3, 8, 6]], dtype=torch.int32)
    hg = hidden.to(DEV).requires_grad_(True)
    eg = embedding.to(DEV).requires_grad_(True)
    value = tiled_tied_cross_entropy(hg, eg, targets.to(DEV), semantic_vocab_size=11, vocab_tile_size=7)
    value.backward()
    h2 = hidden.clone().requires_grad_(True)
    e2 = embedding.clone().requires_grad_(True)
    oracle = oflce.dense_losses(h2, e2, targets, 11, torch.bfloat16).mean()
    oracle.backward()
    print(f"width 5: gpu {float(value):.6f} dense {float(oracle):.6f}", flush=True)
    assert abs(float(value) - float(oracle)) <= 4e-3 + 4e-3 * abs(float(oracle))
    assert value.dtype == torch.float32
    assert hg.grad.dtype == torch.bfloat16 and eg.grad.dtype == torch.float32
    assert tuple(hg.grad.shape) == (2, 3, 5) and tuple(eg.grad.shape) == (13, 5)
    assert maxabs(hg.grad, h2.grad) <= 2e-2 * float(h2.grad.float().abs().max())
    assert maxabs(eg.grad, e2.grad) <= 2e-2 * float(e2.grad.abs().max())
    assert (eg.grad[11:] == 0).all()


def test_float32_compute_reference_fixture():
    """compute_dtype=float32 (rig/kernels/linear_cross_entropy.py:38-41) on
    the reference's own float32 cases (tests/test_linear_cross_entropy.py:
    84-127): hidden (2, 3, 5) from default_rng(7), embedding (13, 5) from
    default_rng(11), semantic vocabulary 11, tile 4; per-token losses within
    rtol = atol = 2e-6 of the dense float32 oracle, the mean and both
    gradients within 3e-6, storage-only rows' gradient exactly zero."""
    from gptrig.kernels import tiled_tied_cross_entropy, tiled_tied_cross_entropy_losses

    hidden = torch.from_numpy(np.random.default_rng(7).normal(size=(2, 3, 5)).astype(np.float32))
    embedding = torch.from_numpy(np.random.default_rng(11).normal(size=(13, 5)).astype(np.float32))
    targets = torch.tensor([[0, 1, 10], [3, 8, 6]], dtype=torch.int32)
    print("flce float32 compute, reference fixture", flush=True)
    losses = tiled_tied_cross_entropy_losses(hidden.to(DEV), embedding.to(DEV), targets.to(DEV),
                                             semantic_vocab_size=11, vocab_tile_size=4, compute_dtype=torch.float32)
    want = oflce.dense_losses(hidden, embedding, targets, 11, torch.float32)
    np.testing.assert_allclose(losses.cpu().numpy(), want.numpy(), rtol=2e-6, atol=2e-6)
    hg = hidden.to(DEV).requires_grad_(True)
    eg = embedding.to(DEV).requires_grad_(True)
    value = tiled_tied_cross_entropy(hg, eg, targets.to(DEV), semantic_vocab_size=11, vocab_tile_size=4,
                                     compute_dtype=torch.float32)
    value.backward()
    h2 = hidden.clone().requires_grad_(True)
    e2 = embedding.clone().requires_grad_(True)
    dense = oflce.dense_losses(h2, e2, targets, 11, torch.float32).mean()
    dense.backward()
    print(f"  gpu {float(value):.8f} dense {float(dense):.8f}", flush=True)
    assert abs(float(value) - float(dense)) <= 2e-6 + 2e-6 * abs(float(dense))
    np.testing.assert_allclose(hg.grad.cpu().numpy(), h2.grad.numpy(), rtol=3e-6, atol=3e-6)
    np.testing.assert_allclose(eg.grad.cpu().numpy(), e2.grad.numpy(), rtol=3e-6, atol=3e-6)
    assert hg.grad.dtype == torch.float32 and eg.grad.dtype == torch.float32
    assert (eg.grad[11:] == 0).all()


@pytest.mark.parametrize("n,d,V,sv,tile", [(300, 96, 1000, 997, 256), (1030, 200, 3001, 2900, 2048), (8, 5, 13, 11, 4)])
def test_float32_compute_matches_float64_dense(n, d, V, sv, tile):
    """The float32 path against the float64 dense closed form at larger,
    ragged shapes (tokens, width, vocabulary and chunks not multiples of the
    64 tile), with invalid targets (+inf loss, no gradient) and per-token
    cotangents: losses to 2e-6 relative, gradients to 1e-5 of their scale."""
    from gptrig.kernels import tiled_tied_cross_entropy_losses

    g = torch.Generator().manual_seed(91)
    h = torch.randn((n, d), generator=g)
    w = torch.randn((V, d), generator=g) * 0.3
    t = torch.randint(0, sv, (n,), generator=g, dtype=torch.int32)
    t[::17] = -1
    ct = torch.rand(n, generator=g)
    print(f"flce float32 compute n={n} d={d} V={V} sv={sv} tile={tile}", flush=True)
    hg = h.to(DEV).requires_grad_(True)
    wg = w.to(DEV).requires_grad_(True)
    losses = tiled_tied_cross_entropy_losses(hg, wg, t.to(DEV), semantic_vocab_size=sv, vocab_tile_size=tile,
                                             compute_dtype=torch.float32)
    finite = torch.isfinite(losses)
    (losses[finite] * ct.to(DEV)[finite]).sum().backward()
    h64 = h.double().requires_grad_(True)
    w64 = w.double().requires_grad_(True)
    logits = h64 @ w64[:sv].t()
    valid = t >= 0
    lse = torch.logsumexp(logits, -1)
    ref = torch.full((n,), float("inf"), dtype=torch.float64)
    ref[valid] = lse[valid] - logits[valid].gather(1, t[valid].long()[:, None])[:, 0]
    (ref[valid] * ct.double()[valid]).sum().backward()
    lc = losses.detach().cpu().double()
    assert torch.equal(torch.isfinite(lc), valid)
    rel = ((lc[valid] - ref[valid]).abs() / ref[valid].abs()).max()
    print(f"  loss rel {float(rel):.2e}", flush=True)
    assert float(rel) <= 2e-6
    for got, want in ((hg.grad, h64.grad), (wg.grad, w64.grad)):
        err = float((got.cpu().double() - want).abs().max())
        scale = float(want.abs().max())
        print(f"  grad max-abs {err:.3e} of {scale:.3e}", flush=True)
        assert err <= 1e-5 * scale
    assert (wg.grad[sv:] == 0).all()


@pytest.mark.parametrize("n,d,V,sv,tile,offset", [
    (1, 1, 1, 1, 1, 0),            # one element everywhere
    (127, 16, 129, 128, 64, 0),    # one row short of / past the 128 tile, one k stage, a 64-row chunk
    (128, 132, 256, 256, 128, 0),  # whole tiles, k = 8 stages and 4 columns
    (129, 37, 385, 300, 200, 0),   # odd width (element loads), ragged chunks
    (514, 64, 1100, 1100, 2048, 1),  # 16-byte loads ruled out by the base address; sliced partial sums
    (1280, 128, 2048, 2000, 1024, 0),  # several slices of both products, two chunks
    (16, 17, 60, 60, 64, 0),       # sums of 16 (multiply-adds), 17 and 60 (eight terms)
    (65, 200, 300, 300, 64, 0),    # sums of 65 and 200 (six terms) beside 64 and 44
    (150, 144, 200, 190, 256, "worst"),  # operands whose dropped terms are the largest
])
def test_float32_split_products_at_tile_edges(n, d, V, sv, tile, offset):
    """The split-operand float32 tiles against float64 where they can go
    wrong: tile, stage, slice and chunk edges, widths and bases without
    16-byte loads, accumulation into dweight, and the same bits twice.

    Bound: a product drops less than 2^-21 of itself (two terms of pieces below
    2^-7 and 2^-15 of their operands) and the operands are split exactly; a sum
    over k is rounded at most six times per 16 products, so an output is within
    (2^-21 + ceil(k/16) 6 2^-24) of the sum of its products' magnitudes, k the
    contraction's length; G adds the error of its logits."""
    from gptrig.kernels import linear_cross_entropy as lce

    g = torch.Generator().manual_seed(n)
    flat = torch.randn(n * d + V * d + 1, generator=g).to(DEV)
    worst = offset == "worst"
    if worst:
        offset, flat = 0, torch.sign(flat) * (1 + 0xFFFF * 2.0 ** -23)
    h = flat[offset:offset + n * d].view(n, d)
    w = flat[offset + n * d:offset + n * d + V * d].mul_(0.25 if worst else 0.3).view(V, d)
    t = torch.randint(0, sv, (n,), generator=g, dtype=torch.int32).to(DEV)
    if n > 5:
        t[3] = -1
        t[5] = sv
    ct = torch.rand(n, generator=g).to(DEV)
    print(f"flce float32 tiles n={n} d={d} V={V} sv={sv} tile={tile} base%16={h.data_ptr() % 16}", flush=True)
    runs = []
    for _ in range(2):
        losses, lse = lce.flce32_forward(h, w, t, sv)
        runs.append((losses, *lce.flce32_backward(h, w, t, lse, ct, 0.0, sv, tile)))
    assert all(torch.equal(a, b) for a, b in zip(*runs))
    losses, dh, dw = (x.cpu().double() for x in runs[0])
    h64, w64, t64 = h.cpu().double(), w.cpu().double(), t.cpu().long()
    valid = (t64 >= 0) & (t64 < sv)
    logits = h64 @ w64[:sv].t()
    lse64 = torch.logsumexp(logits, -1)
    safe = t64.clamp(0, sv - 1)[:, None]
    want = torch.where(valid, lse64 - logits.gather(1, safe)[:, 0], torch.inf)
    c64 = torch.where(valid, ct.cpu().double(), 0.0)[:, None]
    grad = torch.zeros((n, V), dtype=torch.float64)
    grad[:, :sv] = torch.exp(logits - lse64[:, None]) * c64
    grad.scatter_add_(1, safe, -c64)
    eps = lambda k: 2.0 ** -21 + -(-k // 16) * 6 * 2.0 ** -24  # noqa: E731
    # A logit's absolute error; the probabilities (and lse) carry it relatively.
    mags = (h64.abs() @ w64.abs().t()).max()
    dl = float(mags) * eps(d) + 4 * 2.0 ** -24 * float(lse64.abs().max() + 1)
    assert torch.equal(torch.isfinite(losses), valid)
    err = (losses - want)[valid].abs().max()
    print(f"  loss {float(err):.2e} of {2 * dl:.2e}", flush=True)
    assert err <= 2 * dl
    for name, got, ref, big, k in (("dh", dh, grad @ w64, grad.abs() @ w64.abs(), V),
                                   ("dw", dw, grad.t() @ h64, grad.abs().t() @ h64.abs(), n)):
        # (2 dl: the logit's and lse's error; onehot entries keep their own magnitude.)
        p = torch.zeros_like(grad)
        p[:, :sv] = torch.exp(logits - lse64[:, None]) * c64
        noise = p @ w64.abs() if name == "dh" else p.t() @ h64.abs()
        bound = big * eps(k) + noise * (2 * dl + 2.0 ** -22) + 1e-12
        excess = float(((got - ref).abs() / bound).max())
        print(f"  {name} error / bound {excess:.3f}", flush=True)
        assert excess <= 1
    assert (dw[sv:] == 0).all()
    from gptrig import _lib

    base = torch.randn((V, d), generator=g).to(DEV)
    total = base.clone()
    dh2 = torch.empty_like(h)
    ws = _lib.workspace(_lib.query("gptrig_flce32_bwd_workspace_bytes", n, d, V, tile), DEV)
    _lib.call("gptrig_flce32_bwd", h.data_ptr(), w.data_ptr(), t.data_ptr(), lse.data_ptr(), ct.data_ptr(), 0.0,
              dh2.data_ptr(), total.data_ptr(), 1, ws.data_ptr(), ws.numel(), n, d, V, sv, tile, _lib.stream())
    assert torch.equal(dh2, runs[0][1])
    # accumulate_dweight adds to what is there (one more rounding).
    torch.testing.assert_close(total, base + runs[0][2], rtol=0, atol=float(base.abs().max()) * 2.0 ** -22)


def test_float32_tokens_past_one_block():
    """More tokens than one launch addresses (2^22): a whole block and a ragged
    one of 133 tokens, whose rows are padded to 136 columns, against float64.

    Bound as above with k = 8 and 72 for the logits and dh; dw's sum runs over
    the tokens, with a rounding per MFMA and one per block."""
    from gptrig.kernels import linear_cross_entropy as lce

    n, d, V = (1 << 22) + 133, 8, 72
    g = torch.Generator(device=DEV).manual_seed(3)
    h = torch.randn((n, d), generator=g, device=DEV)
    w = torch.randn((V, d), generator=g, device=DEV) * 0.3
    t = torch.randint(0, V, (n,), generator=g, device=DEV, dtype=torch.int32)
    ct = torch.rand(n, generator=g, device=DEV)
    print(f"flce float32 n={n} d={d} V={V}", flush=True)
    losses, lse = lce.flce32_forward(h, w, t, V)
    dh, dw = lce.flce32_backward(h, w, t, lse, ct, 0.0, V, 64)
    dw64 = torch.zeros((V, d), dtype=torch.float64, device=DEV)
    mag64 = torch.zeros_like(dw64)
    w64 = w.double()
    eps = 2.0 ** -20  # of a logit, lse or dh: a few float32 roundings of sums of magnitudes up to ~20
    for i in range(0, n, 1 << 20):
        at = slice(i, i + (1 << 20))
        h64, t64 = h[at].double(), t[at].long()[:, None]
        logits = h64 @ w64.T
        lse64 = torch.logsumexp(logits, -1)
        assert float((lse[at].double() - lse64).abs().max()) <= 16 * eps
        assert float((losses[at].double() - (lse64 - logits.gather(1, t64)[:, 0])).abs().max()) <= 32 * eps
        grad = torch.exp(logits - lse64[:, None]) * ct[at].double()[:, None]
        grad.scatter_add_(1, t64, -ct[at].double()[:, None])
        assert float((dh[at].double() - grad @ w64).abs().max()) <= 32 * eps
        dw64 += grad.T @ h64
        mag64 += grad.abs().T @ h64.abs()
    # (Roundings of a running sum of 2^22 terms: at random signs about the root of their number.)
    excess = float(((dw.double() - dw64).abs() / mag64).max())
    print(f"  dw error / magnitudes {excess:.2e}", flush=True)
    assert excess <= (n // 16) ** 0.5 * 2.0 ** -22


def test_float32_nan_rows_stay_in_their_rows():
    """A NaN hidden row gives a NaN loss and hidden gradient for its token
    alone; the other tokens' losses and hidden gradients are untouched."""
    from gptrig.kernels import linear_cross_entropy as lce

    g = torch.Generator().manual_seed(5)
    h = torch.randn((200, 48), generator=g).to(DEV)
    w = torch.randn((300, 48), generator=g).to(DEV)
    t = torch.randint(0, 300, (200,), generator=g, dtype=torch.int32).to(DEV)
    ct = torch.ones(200, device=DEV)
    print("flce float32 NaN row", flush=True)
    l0, s0 = lce.flce32_forward(h, w, t, 300)
    dh0, _ = lce.flce32_backward(h, w, t, s0, ct, 0.0, 300, 128)
    h[7, 5] = float("nan")
    l1, s1 = lce.flce32_forward(h, w, t, 300)
    dh1, _ = lce.flce32_backward(h, w, t, s1, ct, 0.0, 300, 128)
    rest = torch.arange(200, device=DEV) != 7
    assert torch.isnan(l1[7]) and torch.isnan(dh1[7]).all()
    assert torch.equal(l0[rest], l1[rest]) and torch.equal(dh0[rest], dh1[rest])


@pytest.mark.parametrize("n,d,V,sv,chunk", [
    (8, 64, 40, 33, 8),          # one chunk far below a tile; d not a multiple of 128
    (264, 128, 300, 300, 264),   # one chunk, 8 tokens past a tile
    (520, 192, 700, 650, 256),   # three chunks, the last of 8 tokens
    (600, 128, 1100, 1024, 96),  # chunks below a tile, the last of 24 tokens
    (1032, 256, 513, 513, 512),  # one vocabulary row past two tiles
])
def test_token_chunk_backward_against_float64(n, d, V, sv, chunk):
    """gptrig_flce_bwd_tokens at its edges (chunks and tails that are no token
    tile, ragged vocabularies, storage rows without a class, invalid targets),
    overwriting and accumulating dweight, against float64.

    Bound: bf16 keeps 8 significant bits, so a rounding moves a value by up to
    2^-8 of itself.  Each logit gradient is rounded once (dw: 2^-8 of the sum of
    magnitudes) and dh once more (2^-7 in all); float32 sums, the exponential
    and lse add less than 2^-14."""
    from gptrig import _lib
    from gptrig.kernels import linear_cross_entropy as lce

    g = torch.Generator().manual_seed(n + V)
    h = torch.randn((n, d), generator=g).bfloat16().to(DEV)
    w = (torch.randn((V, d), generator=g) * 0.1).bfloat16().to(DEV)
    t = torch.randint(0, sv, (n,), generator=g, dtype=torch.int32)
    t[1], t[5] = -1, sv
    t = t.to(DEV)
    ct = torch.rand(n, generator=g).to(DEV)
    _, lse = lce.flce_forward(h, w, t, sv)
    print(f"flce token chunks n={n} d={d} V={V} sv={sv} chunk={chunk}", flush=True)
    ws = _lib.workspace(_lib.query("gptrig_flce_bwd_tokens_workspace_bytes", n, d, V, chunk), DEV)
    base = torch.randn((V, d), generator=g).to(DEV)
    got = []
    for accumulate in (0, 1):
        dh = torch.full((n, d), float("nan"), dtype=torch.bfloat16, device=DEV)
        dw = base.clone() if accumulate else torch.full((V, d), float("nan"), device=DEV)
        _lib.call("gptrig_flce_bwd_tokens", h.data_ptr(), w.data_ptr(), t.data_ptr(), lse.data_ptr(), ct.data_ptr(),
                  0.0, dh.data_ptr(), dw.data_ptr(), accumulate, ws.data_ptr(), ws.numel(), n, d, V, sv, chunk,
                  _lib.stream())
        got.append((dh, dw - base if accumulate else dw))
    h64, w64, t64 = h.double(), w.double(), t.long()
    valid = (t64 >= 0) & (t64 < sv)
    logits = h64 @ w64[:sv].T
    c = torch.where(valid, ct.double(), 0.0)[:, None]
    grad = torch.zeros((n, V), dtype=torch.float64, device=DEV)
    grad[:, :sv] = torch.softmax(logits, -1) * c
    grad.scatter_add_(1, t64.clamp(0, sv - 1)[:, None], -c)
    for dh, dw in got:
        for name, x, ref, mag, eps in (("dh", dh, grad @ w64, grad.abs() @ w64.abs(), 2.0 ** -7),
                                       ("dw", dw, grad.T @ h64, grad.abs().T @ h64.abs(), 2.0 ** -8)):
            excess = float(((x.double() - ref).abs() / ((eps + 2.0 ** -14) * mag + 1e-6)).max())
            print(f"  {name} error / bound {excess:.3f}", flush=True)
            assert excess <= 1
    assert (got[0][1][sv:] == 0).all()


def test_public_backward_of_a_very_large_vocabulary():
    """The default public call past the rows whose 32-token blocks stay
    addressable (4,793,481): dh of every token of a 256-token tile and dw, against
    float64 (in slices of the vocabulary); 2^-7 of the magnitudes (two bf16
    roundings) as above."""
    from gptrig.kernels import linear_cross_entropy as lce

    n, d, V = 256, 64, 4_793_481 + 100
    g = torch.Generator(device=DEV).manual_seed(9)
    h = torch.randn((n, d), generator=g, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn((V, d), generator=g, device=DEV) * 0.3).bfloat16().requires_grad_()
    t = torch.randint(0, V, (n,), generator=g, device=DEV, dtype=torch.int32)
    assert lce.token_chunk(n, d, V, lce.chunk_for(2048)) == 0
    print(f"flce public backward n={n} d={d} V={V}", flush=True)
    lce.tiled_tied_cross_entropy(h, w, t, semantic_vocab_size=V).backward()
    h64, t64 = h.detach().double(), t.long()
    cut = [slice(i, min(i + (1 << 17), V)) for i in range(0, V, 1 << 17)]
    lse = torch.logsumexp(torch.stack([torch.logsumexp(h64 @ w.detach()[c].double().T, -1) for c in cut], -1), -1)
    dh, mag, worst = torch.zeros_like(h64), torch.zeros_like(h64), 0.0
    for c in cut:
        w64 = w.detach()[c].double()
        grad = torch.exp(h64 @ w64.T - lse[:, None]) / n
        mine = ((t64 >= c.start) & (t64 < c.stop)).nonzero()[:, 0]
        grad[mine, t64[mine] - c.start] -= 1.0 / n
        dh += grad @ w64
        mag += grad.abs() @ w64.abs()
        bound = 2.0 ** -7 * (grad.abs().T @ h64.abs()) + 1e-9
        worst = max(worst, float(((w.grad[c].double() - grad.T @ h64).abs() / bound).max()))
    excess = float(((h.grad.double() - dh).abs() / (2.0 ** -7 * mag + 1e-9)).max())
    print(f"  error / bound: dh {excess:.3f}, dw {worst:.3f}", flush=True)
    assert excess <= 1 and worst <= 1


def test_token_chunk_backward_of_a_new_count_costs_no_more_on_the_host():
    """A token count the process has not seen before is planned as quickly as a
    known one: the host's time of the first call over that of the second, median
    over 24 counts, below 100 us (walking the plan's items took 400 us and
    more)."""
    import time

    from gptrig import _lib
    from gptrig.kernels import linear_cross_entropy as lce

    d, V, n_max = 128, 50304, 24 * 256 + 2048
    h = torch.randn((n_max, d), device=DEV).bfloat16()
    w = (torch.randn((V, d), device=DEV) * 0.1).bfloat16()
    t = torch.zeros(n_max, dtype=torch.int32, device=DEV)
    lse, dh, dw = torch.full((n_max,), 11.0, device=DEV), torch.empty_like(h), torch.empty((V, d), device=DEV)
    ws = _lib.workspace(_lib.query("gptrig_flce_bwd_tokens_workspace_bytes", n_max, d, V, n_max), DEV)

    def host_us(n):
        torch.cuda.synchronize()
        start = time.perf_counter()
        _lib.call("gptrig_flce_bwd_tokens", h.data_ptr(), w.data_ptr(), t.data_ptr(), lse.data_ptr(), None, 1e-3,
                  dh.data_ptr(), dw.data_ptr(), 0, ws.data_ptr(), ws.numel(), n, d, V, V, n, _lib.stream())
        return (time.perf_counter() - start) * 1e6

    host_us(n_max)
    extra = sorted(host_us(n) - host_us(n) for n in range(2048, n_max - 255, 256))
    print(f"flce new token counts: first call over second {extra[12]:.0f} us (median of {len(extra)})", flush=True)
    assert extra[12] < 100


def test_public_backward_route_and_memory():
    """The token chunk the public call takes: within the memory it may use,
    whole tokens where they fit, and none for a tile below the default (whose
    gradients agree with the default's)."""
    from gptrig import _lib
    from gptrig.kernels import linear_cross_entropy as lce

    V = 50304
    for n in (8, 128, 1000, 4096, 16384, 65536):
        for d in (64, 512, 576, 768, 1024):
            for tile in (256, 1792, 2048, 4096, V + 256):
                chunk = lce.token_chunk(n, d, V, lce.chunk_for(tile))
                if tile < 2048:
                    assert chunk == 0
                elif chunk:
                    assert chunk == n or (chunk < n and chunk % 256 == 0)
                    assert _lib.query("gptrig_flce_bwd_tokens_workspace_bytes", n, d, V, chunk) <= max(
                        4 * n * lce.chunk_for(tile), 4 * V * d * 17 // 16)
    assert lce.token_chunk(128, 768, V, 2048) == 128 and lce.token_chunk(16384, 768, V, 2048) % 256 == 0
    g = torch.Generator().manual_seed(3)
    h, w = torch.randn((300, 72), generator=g).to(DEV), (torch.randn((5000, 72), generator=g) * 0.1).to(DEV)
    t = torch.randint(0, 4990, (300,), generator=g, dtype=torch.int32).to(DEV)
    print("flce public route: default tile against 512", flush=True)
    grads = []
    for tile in (2048, 512):
        hg, wg = h.clone().requires_grad_(), w.clone().requires_grad_()
        lce.tiled_tied_cross_entropy(hg, wg, t, semantic_vocab_size=4990, vocab_tile_size=tile).backward()
        grads.append((hg.grad, wg.grad))
    for a, b in zip(*grads):  # one bf16 rounding of dh apart at most
        assert float((a - b).norm()) <= 2.0 ** -9 * float(b.norm())


@pytest.mark.parametrize("n,d,V,tile", [(200, 48, 300, 128), (130, 37, 257, 2048)])
def test_float32_infinite_operands(n, d, V, tile):
    """Infinite weights and activations give what float32 products give: a
    class of -inf weights drops out of the sum over positive activations, an
    infinite activation makes its own token's results infinite or NaN, and the
    products past the largest float32 are infinities.  Finite values as in the
    other float32 tests (1e-5)."""
    from gptrig.kernels import linear_cross_entropy as lce

    g = torch.Generator().manual_seed(n)
    h = (torch.rand((n, d), generator=g) + 0.1).to(DEV)
    w = (torch.randn((V, d), generator=g) * 0.3).to(DEV)
    w[10] = w[130] = -torch.inf
    w[11, 3] = -torch.inf
    h[7, 5] = torch.inf
    h[9] = 1e30
    w[12] = -1e30  # (-inf as a product of finite operands, for token 9)
    t = torch.randint(20, 120, (n,), generator=g, dtype=torch.int32).to(DEV)
    ct = torch.rand(n, generator=g).to(DEV)
    print(f"flce float32 infinities n={n} d={d} V={V}", flush=True)
    losses, lse = lce.flce32_forward(h, w, t, V)
    dh, dw = lce.flce32_backward(h, w, t, lse, ct, 0.0, V, tile)
    logits = (h.double()[:, None, :] * w.double()[None]).sum(-1)
    fine = torch.ones(n, dtype=torch.bool, device=DEV)
    fine[7] = False
    want_lse = torch.logsumexp(logits, -1)
    want = want_lse - logits.gather(1, t.long()[:, None])[:, 0]
    assert torch.isfinite(want[fine]).all()
    assert float(((losses.double() - want).abs() / (want.abs() + 1))[fine].max()) <= 1e-5
    assert not torch.isfinite(losses[7])
    # dw of the classes from the other tokens (without 9, whose 1e30 hides them).
    fine[9] = False
    keep = fine.nonzero()[:, 0]
    _, dw2 = lce.flce32_backward(h[keep].contiguous(), w, t[keep].contiguous(), lse[keep].contiguous(),
                                 ct[keep].contiguous(), 0.0, V, tile)
    grad = torch.exp(logits[keep] - want_lse[keep, None])
    grad[torch.arange(len(keep), device=DEV), t[keep].long()] -= 1
    want_dw = (grad * ct[keep, None].double()).T @ h[keep].double()
    assert torch.isfinite(want_dw).all() and (want_dw[10] == 0).all() and (dw2[10] == 0).all()
    assert float((dw2.double() - want_dw).abs().max()) <= 1e-5 * float(want_dw.abs().max())
    # dh is 0 x -inf where a class of -inf weights has probability 0, as in a float32 product.
    assert torch.isnan(dh[fine]).any(1).all() and torch.isnan(dw[20:120]).any()


@pytest.mark.parametrize("n,d,positive", [
    (1, 4, False), (2, 8, False), (4, 16, False), (9, 32, False), (17, 200, False), (129, 64, False),
    (65, 70, False), (4, 16, True), (64, 24, True), (65, 66, True), (140, 140, True),
])
def test_float32_products_are_no_less_precise_than_a_chain(n, d, positive):
    """Both gradients' errors against float64 next to those of one float32
    multiply-add chain per output (from the same log-sum-exp), over short and
    long sums, operands of random signs and of one sign.  Errors are random: over
    these draws the ratio of their root mean squares spreads by about a tenth, so
    1.15 for random signs; 1.35 for one sign, where the matrix cores' roundings
    share theirs (without the two further terms, the short sums' multiply-adds and
    the small terms' accumulator: 1.9 to 2.3)."""
    from gptrig.kernels import linear_cross_entropy as lce

    V, draws = 400, 48 if n <= 4 else 12

    def chain(a, b):
        acc = torch.zeros((a.shape[0], b.shape[1]), dtype=torch.float64, device=DEV)
        for k in range(a.shape[1]):  # a float64 product of two float32 is exact
            acc = (acc + a[:, k, None].double() * b[k].double()).float().double()
        return acc

    def grad(logits, lse, t, ct):
        g = torch.exp(logits - lse[:, None])
        g[torch.arange(n, device=DEV), t.long()] -= 1
        return g * ct[:, None]

    print(f"flce float32 precision n={n} d={d} positive={positive}", flush=True)
    err = torch.zeros(4, dtype=torch.float64)
    for seed in range(draws):
        g = torch.Generator(device=DEV).manual_seed(seed)
        h = torch.randn((n, d), generator=g, device=DEV)
        w = torch.randn((V, d), generator=g, device=DEV) * 0.3
        if positive:
            h.abs_(), w.abs_()
        t = torch.randint(0, V, (n,), generator=g, device=DEV, dtype=torch.int32)
        ct = torch.rand(n, generator=g, device=DEV)
        l64 = h.double() @ w.double().T
        g64 = grad(l64, torch.logsumexp(l64, -1), t, ct.double())
        _, lse = lce.flce32_forward(h, w, t, V)
        gc = grad(chain(h, w.T.contiguous()).float(), lse, t, ct)
        dh, dw = lce.flce32_backward(h, w, t, lse, ct, 0.0, V, 2048)
        for i, (got, want) in enumerate(((dw, g64.T @ h.double()), (chain(gc.T.contiguous(), h), g64.T @ h.double()),
                                         (dh, g64 @ w.double()), (chain(gc, w), g64 @ w.double()))):
            err[i] += float(((got.double() - want).norm() / want.norm()) ** 2)
    dw_ratio, dh_ratio = float((err[0] / err[1]).sqrt()), float((err[2] / err[3]).sqrt())
    print(f"  error over the chain's: dw {dw_ratio:.2f}, dh {dh_ratio:.2f}", flush=True)
    assert max(dw_ratio, dh_ratio) <= (1.35 if positive else 1.15)


def test_float32_chunk_rows_follow_the_tile_and_the_weight_gradient():
    """The float32 backward's chunk: the tile itself below the default,
    otherwise at least the tile, and the logit gradient within the tile's or half
    the weight gradient's size; one short call through the larger chunk."""
    from gptrig.kernels import linear_cross_entropy as lce

    V = 50304
    for n in (1, 128, 2048, 16384):
        for d in (5, 64, 512):
            for tile in (1, 2047, 2048, 4096, 10 * V):
                rows = lce.vocab_rows32(n, d, V, tile)
                assert rows == tile if tile < 2048 else rows >= tile
                assert rows <= max(tile, V) and (rows == tile or 4 * n * rows <= 2 * V * d)
    g = torch.Generator().manual_seed(8)
    h, w = torch.randn((40, 48), generator=g).to(DEV), torch.randn((4500, 48), generator=g).to(DEV)
    t = torch.randint(0, 4400, (40,), generator=g, dtype=torch.int32).to(DEV)
    print("flce float32 default tile (two chunks' worth of rows) against 1024", flush=True)
    grads = []
    for tile in (2048, 1024):
        hg, wg = h.clone().requires_grad_(), w.clone().requires_grad_()
        lce.tiled_tied_cross_entropy(hg, wg, t, semantic_vocab_size=4400, vocab_tile_size=tile,
                                     compute_dtype=torch.float32).backward()
        grads.append((hg.grad, wg.grad))
    for a, b in zip(*grads):  # the same float32 sums in another order
        assert float((a - b).norm()) <= 1e-6 * float(b.norm())
