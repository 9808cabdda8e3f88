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
