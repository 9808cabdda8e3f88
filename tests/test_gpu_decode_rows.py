"""GPU: segments of every height around the gate/up kernel's staging limits (rows that fit the LDS in one pass, in two,
in four; one or two staged matrices; duplicated rows), against the oracle at the kernel's rounding points (fp32 sums in
another order: rel_l2 <= 5e-4, as for the other decode cases)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe, routing

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _check(cuda, K, N, rows, **suh):
    from mi355moe import _lib, ops, synthetic
    print(f"decode rows={rows} K={K} N={N} {suh}", flush=True)
    n, topk = 5, 2
    ex = synthetic.calibrated_layer(n, K, N, seed=11, device=cuda, **suh)
    x = synthetic.activations(rows, K, seed=12, device=cuda)
    ids = torch.stack([torch.zeros(rows, dtype=torch.int32), 1 + torch.arange(rows, dtype=torch.int32) % 4], 1).to(cuda)
    w = synthetic.softmax_weights(rows, topk, seed=13, device=cuda)
    got = ops.moe_forward_ids(ex, x, ids, w, out_dtype=torch.float32, path=_lib.PATH_DECODE).cpu().numpy()
    lay = {k: getattr(ex, k).cpu().numpy() for k in ("w13_trellis", "w13_suh", "w13_svh", "w2_trellis", "w2_suh",
                                                     "w2_svh")}
    tok, e, w16 = moe.pairs_from_routing(routing.map_topk_to_local(ids.cpu().numpy(), n, None), w.cpu().numpy(), n, topk)
    ref = moe.forward(lay, x.cpu().to(torch.float16).numpy(), tok, e, w16, 10.0, "decode_x")
    assert np.isfinite(got).all()
    assert _rel(got, ref) <= 5e-4


@pytest.mark.parametrize("K,N,shared", [(4096, 256, True), (4096, 128, False), (8192, 128, True), (6144, 128, True),
                                        (1024, 384, False)])
@pytest.mark.parametrize("rows", [1, 4, 5, 8, 9, 15, 16, 17, 35])
def test_rows_per_segment(cuda, K, N, shared, rows):
    _check(cuda, K, N, rows, shared_suh=shared)


# hidden sizes that are odd multiples of 256 have no halves: rows that pass the two-per-CU LDS limit are staged whole
@pytest.mark.parametrize("K,shared,rows", [(2560, True, 16), (2816, True, 8), (2816, True, 16), (4864, True, 16),
                                           (4864, True, 33), (1792, False, 16), (2304, False, 9)])
def test_rows_of_odd_hidden(cuda, K, shared, rows):
    _check(cuda, K, 128, rows, shared_suh=shared)
    if shared:
        _check(cuda, K, 128, rows, uniform_suh=True)


# one w13 suh for every expert: calls of more than 4 rows rotate them once per token (with the call's first route launch,
# or, GATEUP staged alone, in a launch of its own) and the workgroups copy them, by LDS DMA where a pass is whole 512-k pieces, by register loads where it is not or where the rows are duplicated
@pytest.mark.parametrize("K,N", [(4096, 256), (8192, 128), (6144, 128), (768, 128), (256, 128), (10240, 128)])
@pytest.mark.parametrize("rows", [3, 4, 5, 9, 16, 17, 35, 520])
def test_rows_rotated_once(cuda, K, N, rows):
    _check(cuda, K, N, rows, uniform_suh=True)


@pytest.mark.parametrize("rows", [5, 40])
def test_rows_rotated_by_stage(cuda, rows):
    """The routing staged alone, then the experts (whose rotation is then a launch of its own): bit-equal to one call."""
    from mi355moe import _lib, ops, synthetic
    print(f"decode by stage rows={rows}", flush=True)
    ex = synthetic.calibrated_layer(5, 1280, 128, seed=11, device=cuda, uniform_suh=True)
    x = synthetic.activations(rows, 1280, seed=12, device=cuda)
    ids = torch.stack([torch.zeros(rows, dtype=torch.int32), 1 + torch.arange(rows, dtype=torch.int32) % 4], 1).to(cuda)
    w = synthetic.softmax_weights(rows, 2, seed=13, device=cuda)
    kw = dict(out_dtype=torch.float32, path=_lib.PATH_DECODE)
    whole = ops.moe_forward_ids(ex, x, ids, w, **kw)
    out = torch.zeros_like(whole)
    ops.moe_forward_ids(ex, x, ids, w, out=out, stages=_lib.STAGE_ROUTE, **kw)
    ops.moe_forward_ids(ex, x, ids, w, out=out, stages=_lib.STAGE_GATEUP | _lib.STAGE_DOWN | _lib.STAGE_COMBINE, **kw)
    assert torch.equal(out, whole)
