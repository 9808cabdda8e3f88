"""GPU: one expert-parallel rank of a layer on the grouped tier. Its tile kind follows the pairs expected on its own
experts, and the combine skips the slots of other ranks; both are bit-identical to the 256-row tiles over the same
routing, and the output matches the oracle (rel_l2 <= 5e-4, the bar of the other grouped cases)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe, routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,topk,local", [(300, 4, 8), (300, 4, 1), (257, 9, 4), (130, 1, 2)])
def test_rank(cuda, monkeypatch, T, topk, local):
    from mi355moe import _lib, ops, synthetic
    n_global, K, N = 16, 512, 256
    print(f"ep rank T={T} topk={topk} local={local} of {n_global}", flush=True)
    ex = synthetic.calibrated_layer(local, K, N, seed=21, device=cuda, uniform_suh=True)
    x = synthetic.activations(T, K, seed=22, device=cuda)
    g = torch.Generator().manual_seed(23)
    ids = torch.rand(T, n_global, generator=g).topk(topk, 1).indices.to(torch.int32).to(cuda)
    w = synthetic.softmax_weights(T, topk, seed=24, device=cuda)
    emap = torch.full((n_global,), -1, dtype=torch.int64)
    emap[3:3 + local] = torch.arange(local)                          # tokens without a local expert among them
    got = {}
    for tiles in ("auto", "large"):
        monkeypatch.setenv("MI355MOE_PREFILL_TILES", tiles)
        got[tiles] = ops.moe_forward_ids(ex, x, ids, w, out_dtype=torch.float32, expert_map=emap.to(cuda),
                                         path=_lib.PATH_PREFILL).cpu().numpy()
    assert np.array_equal(got["auto"], got["large"])
    lay = {k: getattr(ex, k).cpu().numpy() for k in ("w13_trellis", "w13_suh", "w13_svh", "w2_trellis", "w2_suh",
                                                     "w2_svh")}
    tok, e, w16 = moe.pairs_from_routing(routing.map_topk_to_local(ids.cpu().numpy(), local, emap.numpy()),
                                         w.cpu().numpy(), local, topk)
    ref = moe.forward(lay, x.cpu().to(torch.float16).numpy(), tok, e, w16, 10.0, "e3")
    assert np.linalg.norm(got["auto"] - ref) <= 5e-4 * np.linalg.norm(ref)


@pytest.mark.parametrize("T", [1, 8, 15])
def test_rank_decode(cuda, T):
    """Decode calls of a rank with 96 of 192 experts: the gate/up reduction splits for the experts the rank reaches."""
    from mi355moe import _lib, ops, synthetic
    n, n_global, K, N, topk = 96, 192, 4096, 256, 8
    print(f"ep rank decode T={T}", flush=True)
    ex = synthetic.calibrated_layer(n, K, N, seed=25, device=cuda, uniform_suh=True)
    x = synthetic.activations(T, K, seed=26, device=cuda)
    ids = torch.rand(T, n_global, generator=torch.Generator().manual_seed(27)).topk(topk, 1).indices.to(torch.int32).to(cuda)
    w = synthetic.softmax_weights(T, topk, seed=28, device=cuda)
    emap = torch.full((n_global,), -1, dtype=torch.int64)
    emap[::2] = torch.arange(n)
    got = ops.moe_forward_ids(ex, x, ids, w, out_dtype=torch.float32, expert_map=emap.to(cuda),
                              path=_lib.PATH_DECODE).cpu().numpy()
    lay = {k: getattr(ex, k).cpu().numpy() for k in ("w13_trellis", "w13_suh", "w13_svh", "w2_trellis", "w2_suh",
                                                     "w2_svh")}
    tok, e, w16 = moe.pairs_from_routing(routing.map_topk_to_local(ids.cpu().numpy(), n, emap.numpy()),
                                         w.cpu().numpy(), n, topk)
    ref = moe.forward(lay, x.cpu().to(torch.float16).numpy(), tok, e, w16, 10.0, "decode_x")
    assert np.linalg.norm(got - ref) <= 5e-4 * np.linalg.norm(ref)


@pytest.mark.parametrize("T,K,N,topk", [(1, 2048, 512, 4), (3, 4096, 1024, 8), (7, 2048, 1024, 6), (24, 4096, 512, 6),
                                        (48, 4096, 256, 8)])
def test_rank_decode_splits(cuda, T, K, N, topk):
    """A rank's call against one call per pick over its local ids (plans of T pairs, with other splits): the same sums in
    another order, within the bar that each keeps to the oracle (rel_l2 <= 5e-4)."""
    from mi355moe import _lib, ops, synthetic
    n = 12
    print(f"ep rank decode splits T={T} K={K} N={N} topk={topk}", flush=True)
    ex = synthetic.calibrated_layer(n, K, N, seed=31, device=cuda, uniform_suh=True)
    x = synthetic.activations(T, K, seed=32, device=cuda)
    ids = torch.rand(T, 8 * n, generator=torch.Generator().manual_seed(33)).topk(topk, 1).indices.to(torch.int32)
    ids[:, 0] = torch.arange(T, dtype=torch.int32) % n               # every token has a local expert
    ids[:, 1:] += (ids[:, 1:] == ids[:, :1]).int() * n               # (distinct picks)
    w = synthetic.softmax_weights(T, topk, seed=34, device=cuda)
    emap = torch.full((8 * n + n,), -1, dtype=torch.int64)
    emap[:n] = torch.arange(n)
    kw = dict(out_dtype=torch.float32, path=_lib.PATH_DECODE)
    got = ops.moe_forward_ids(ex, x, ids.to(cuda), w, expert_map=emap.to(cuda), **kw)
    here = (ids < n).to(cuda)
    ref = torch.zeros_like(got)
    for k in range(topk):                                            # one pick at a time: plans of T pairs
        one = torch.where(here[:, k:k + 1], ids[:, k:k + 1].to(cuda), -1)
        ref += ops.moe_forward_ids(ex, x, one.int().contiguous(), w[:, k:k + 1].contiguous(), **kw)
    assert float((got - ref).norm()) <= 5e-4 * float(ref.norm())
