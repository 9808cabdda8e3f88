"""GPU: the whole-layer call's picks and weights, which come from bounded logits with the exact dot product only where a
bound wins a round, against the exact logits ranked by themselves (bit-exact), over token and expert counts around the
tile edges, every K split, equal logits, and operands whose fp32 sums or norms hold nothing."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(cuda, T, E, K, topk, x, w, b, renorm=True):
    from mi355moe import ops, synthetic
    ex = synthetic.exl3_layer(2, K, 128, seed=3, device=cuda)
    lg = ops.router_logits(x, w)
    ids, wts = ops.router_topk(lg, topk, bias=b, routed_scale=2.5, renormalize=renorm)
    _, gi, gw = ops.moe_layer(ex, x, router_w=w, topk=topk, bias=b, routed_scale=2.5, renormalize=renorm,
                              return_picks=True)
    torch.cuda.synchronize()
    assert torch.equal(ids, gi)
    assert torch.equal(wts.view(torch.int32), gw.view(torch.int32))


@pytest.mark.parametrize("T,E,K,topk", [(17, 288, 4096, 8), (31, 33, 512, 4), (33, 32, 1024, 32), (64, 288, 4096, 8),
                                        (65, 1, 2048, 1), (130, 65, 8192, 6), (257, 320, 4096, 8), (300, 321, 512, 8),
                                        (1025, 1024, 1024, 8), (4097, 288, 4096, 8)])
def test_picks_equal_exact_logits(cuda, T, E, K, topk):
    print(f"picks T={T} E={E} K={K} topk={topk}", flush=True)
    from mi355moe import synthetic
    w, b = synthetic.router(E, K, seed=5, device=cuda)
    x = synthetic.activations(T, K, seed=6, device=cuda)
    _check(cuda, T, E, K, topk, x, w, b)
    _check(cuda, T, E, K, topk, x, w, None, renorm=False)


@pytest.mark.parametrize("kind", ["ties", "tiny", "huge", "zero", "outliers", "nan"])
def test_picks_hard_operands(cuda, kind):
    print(f"picks operands {kind}", flush=True)
    from mi355moe import synthetic
    T, E, K = 70, 288, 4096
    w, b = synthetic.router(E, K, seed=7, device=cuda)
    x = synthetic.activations(T, K, seed=8, device=cuda)
    if kind == "ties":                                # every logit four times, biases equal: the lowest ids win
        w = w[: E // 4].repeat(4, 1).contiguous()
        b = torch.zeros_like(b)
    elif kind == "tiny":                              # squares below the fp32 range
        x = x * 1e-24
    elif kind == "huge":                              # squares beyond it; sigmoids at 0 and 1
        x = x * 1e22
    elif kind == "zero":
        x[:35] = 0
    elif kind == "outliers":
        x[:, ::512] *= 3000.0
    elif kind == "nan":
        x[3, 5], x[4, 6], x[5, 7], w[9, 5] = float("nan"), float("inf"), -float("inf"), 0.0
    _check(cuda, T, E, K, 8, x, w, b)


def _operands(cuda, kind, T, E, K):
    from mi355moe import synthetic
    w, b = synthetic.router(E, K, seed=17, device=cuda)
    x = synthetic.activations(T, K, seed=18, device=cuda)
    g = torch.Generator(device=cuda).manual_seed(19)
    if kind == "zero":                                # padding: token rows and experts
        x[::2] = 0
        w[1::3] = 0
    elif kind == "tiny":                              # squares below the fp32 range; scores all 0.5
        x[::2] *= 1e-22
        w[1::3] *= 1e-20
    elif kind == "huge":                              # norms past the fp32 range, half of the tokens and one expert
        x[::2] *= 1e25
        w[3] *= 1e30
    elif kind == "nan":
        x[T - 2, 5], x[7, K - 1], w[E - 1, 3] = float("nan"), float("inf"), float("nan")
    elif kind == "cancel":                            # sums far below the norms: whole and in every pair of products
        x[:, 1::2] = x[:, ::2]
        w[:, 1::2] = -w[:, ::2]
        w += (torch.randn(E, K, generator=g, device=cuda) * 1e-4).to(w.dtype)
    elif kind == "wide":                              # exponents over 24 binades
        x *= torch.exp2(torch.rand(T, K, generator=g, device=cuda) * 24 - 12).to(x.dtype)
        w *= torch.exp2(torch.rand(E, K, generator=g, device=cuda) * 24 - 12).to(w.dtype)
    elif kind == "outliers":                          # a few large channels that the router weights down
        x[:, ::512] *= 300.0
        w[:, ::512] *= 0.003
    return x, w, b


# the small tiles, and from 1024 tokens the large ones; up to 320 experts and more (another top-k); partial tiles
@pytest.mark.parametrize("T,E,K", [(33, 40, 1024), (70, 288, 4096), (1030, 100, 512), (1100, 400, 2048)])
@pytest.mark.parametrize("kind", ["plain", "zero", "tiny", "huge", "nan", "cancel", "wide", "outliers"])
def test_bound_words(cuda, kind, T, E, K):
    """Every stored word against the exact logit: exact ones are it (or 0 for one within 2^-26, whose score is 0.5 too),
    upper bounds are not below it, and rows that are zero, tiny, not finite or too large for fp32 norms have exact words
    only. The picks and weights are those of the exact logits."""
    import ctypes

    from mi355moe import _lib, ops, synthetic
    print(f"bound words {kind} T={T} E={E} K={K}", flush=True)
    topk = 8
    x, w, b = _operands(cuda, kind, T, E, K)
    ex = synthetic.exl3_layer(2, K, 128, seed=3, device=cuda)
    lg = ops.router_logits(x, w)
    ids, wts = ops.router_topk(lg, topk, bias=b, routed_scale=2.5)
    _, gi, gw = ops.moe_layer(ex, x, router_w=w, topk=topk, bias=b, routed_scale=2.5, return_picks=True)
    # the call's router scratch follows the experts' part of the workspace
    desc = ctypes.byref(ex.desc)
    base = _lib.lib().mi355moe_moe_workspace_bytes_path(desc, T, topk, _lib.PATH_AUTO)
    ws = ops.workspace(cuda, _lib.lib().mi355moe_moe_layer_workspace_bytes(desc, T, topk, E))
    off = (base + 255) // 256 * 256
    words = ws[off:off + 4 * T * E].view(torch.int32).view(T, E).clone()
    torch.cuda.synchronize()
    low, val = words & 0xFFFF, (words & -65536).view(torch.float32)
    assert ((low == 0) | (low == 1)).all()
    small = lg.abs() <= 2.0 ** -26
    ok = torch.where(low == 0, (val == lg) | (small & (val == 0)) | (val.isnan() & lg.isnan()), val >= lg)
    assert ok.all(), (kind, int((~ok).sum()), lg[~ok][:4], val[~ok][:4])
    known = {"zero": (slice(None, None, 2), slice(1, None, 3)), "tiny": (slice(None, None, 2), slice(1, None, 3)),
             "huge": (slice(None, None, 2), 3), "nan": ([T - 2, 7], E - 1)}.get(kind)
    if known:
        assert (low[known[0]] == 0).all() and (low[:, known[1]] == 0).all()
    assert torch.equal(ids, gi)
    assert torch.equal(wts.view(torch.int32), gw.view(torch.int32))


@pytest.mark.parametrize("T", [40, 1030])
def test_picks_of_unaligned_rows(cuda, T):
    """x a column range of a wider buffer, 8 bytes past a 16-byte address (its row stride is a multiple of 16 bytes)."""
    from mi355moe import synthetic
    print(f"picks of unaligned rows T={T}", flush=True)
    E, K = 100, 1024
    w, b = synthetic.router(E, K, seed=25, device=cuda)
    wide = synthetic.activations(T, K + 64, seed=26, device=cuda)
    x = wide[:, 4:4 + K]
    assert x.data_ptr() % 16 == 8
    _check(cuda, T, E, K, 4, x, w, b)
