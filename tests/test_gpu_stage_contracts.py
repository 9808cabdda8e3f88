"""GPU parity of the stage entry points over caller-built row tables: the grouped (E3) trio with its table builder
and apply (the contracts of code/fork/docs/prod_exl3_reference.py:1316-1435), and the e4m3 extension's stages as the
overlay's run() chains them (code/fork/overlay/glm53_moe_e4m3.py:450-592: plan, gather_tok / gather2, fused, or the
chunked gateup / actq / down), each against the oracle. Tables are compared bit for bit with independent numpy-loop
constructions of the same contracts; the stages' buffers (e4m3 codes in the extension's byte order, row scales, the
SwiGLU output) are compared with the oracle's stage functions, as the reference's own stage checks A1-A4 do
(code/fork/tests/moee4m3/test_moe_e4m3.py:111-181)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import e4m3, e4m3_trellis, moe, routing

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


def _np_layer(ex) -> dict:
    return {k: getattr(ex, k).cpu().numpy() for k in ("w13_trellis", "w13_suh", "w13_svh", "w2_trellis", "w2_suh",
                                                      "w2_svh")}


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("cap", [0, 140, 10 ** 6])
def test_e3_trio_apply(cuda, cap):
    """apply_exl3_grouped_fat over production's routing prelude: out (fp32, pre-filled) += the fat experts' (count >
    cap) routed output; cap 0 = every expert, 10**6 = none (out untouched)."""
    from mi355moe import e3, synthetic
    n, K, N, T, topk = 16, 1024, 512, 300, 8
    _say(f"E3 trio n={n} K={K} N={N} T={T} topk={topk} cap={cap}")
    ex = synthetic.calibrated_layer(n, K, N, seed=5, device=cuda)
    x16 = synthetic.activations(T, K, seed=6, device=cuda).to(torch.float16)
    ids = synthetic.random_ids(T, n, topk, seed=7, device=cuda)
    w = synthetic.softmax_weights(T, topk, seed=8, device=cuda)
    local = ids.reshape(-1).long()
    order = torch.argsort(local, stable=True)
    counts = torch.bincount(local, minlength=n + 1)[:n].contiguous()
    token_sorted = torch.div(order, topk, rounding_mode="floor")
    weight_sorted = w.reshape(-1)[order].to(torch.float16)
    base = torch.randn(T, K, device=cuda) * 0.1
    out = base.clone()
    e3.apply_exl3_grouped_fat(x16, out, counts, token_sorted, weight_sorted, ex, cap, 10.0)
    again = base.clone()
    e3.apply_exl3_grouped_fat(x16, again, counts, token_sorted, weight_sorted, ex, cap, 10.0)
    torch.cuda.synchronize()
    assert torch.equal(out, again)                                 # deterministic (row-order sums, no atomics)
    fat = (counts > cap).cpu().numpy()
    lid = local.cpu().numpy()
    exx = np.where(fat[lid], lid, -1).astype(np.int32)
    tok = (np.arange(T * topk) // topk).astype(np.int32)
    w16 = w.reshape(-1).cpu().numpy().astype(np.float16)
    got = (out - base).cpu().numpy()
    if not fat.any():
        assert not got.any()
        return
    lay = _np_layer(ex)
    xs = x16.cpu().numpy()
    ref_k = moe.forward(lay, xs, tok, exx, w16, 10.0, "e3")
    ref64 = moe.forward(lay, xs, tok, exx, w16, 10.0, "f64_pre")
    r_k, r64 = _rel(got, ref_k), _rel(got, ref64)
    _say(f"  fat experts {int(fat.sum())}/{n}: rel_l2 vs E3 rounding {r_k:.3e}, vs float64 {r64:.3e}")
    assert r_k <= 5e-4 and r64 <= 5e-3
    assert np.allclose(got, ref64, rtol=2e-2, atol=1e-3)


def _fat_tables_loop(counts, cap, token_sorted, weight_sorted, tile):
    """The fat tables by plain loops: experts with more than cap pairs in expert order, their pairs' tokens and
    weights in sorted order, one segment per tile rows."""
    rows, segs = [], []
    start = 0
    for e, c in enumerate(counts):
        c = int(c)
        if c > cap:
            r0 = len(rows)
            for i in range(c):
                rows.append((e, int(token_sorted[start + i]), weight_sorted[start + i]))
            for q in range(0, c, tile):
                segs.append((e, r0 + q, min(tile, c - q)))
        start += c
    return rows, segs


@pytest.mark.parametrize("cap,tile", [(0, 256), (37, 256), (37, 64), (10 ** 6, 256)])
def test_e3_fat_tables_vs_loop(cuda, cap, tile):
    from mi355moe import e3
    g = np.random.default_rng(cap + tile)
    n = 40
    counts = g.integers(0, 90, n)
    counts[::5] = 0
    counts[3] = 700                                                   # several segments
    P = int(counts.sum())
    tok = g.integers(0, 1000, P).astype(np.int64)
    w16 = g.random(P).astype(np.float16)
    rows_cap = P + 17                                                 # capacity beyond the live rows
    tok_c = np.concatenate([tok, np.zeros(17, np.int64)])
    w_c = np.concatenate([w16, np.zeros(17, np.float16)])
    t = e3.build_grouped_fat_tables(torch.from_numpy(counts).to(cuda), cap, torch.from_numpy(tok_c).to(cuda),
                                    torch.from_numpy(w_c).to(cuda), rows_cap, tile)
    rows, segs = _fat_tables_loop(counts, cap, tok, w16, tile)
    nr, ns = int(t["num_rows"].item()), int(t["num_segs"].item())
    assert nr == len(rows) and ns == len(segs)
    if rows:
        assert np.array_equal(t["row_expert"][:nr].cpu().numpy(), [r[0] for r in rows])
        assert np.array_equal(t["row_token"][:nr].cpu().numpy(), [r[1] for r in rows])
        assert np.array_equal(t["row_weight"][:nr].cpu().numpy(), np.array([r[2] for r in rows], np.float16))
        assert np.array_equal(t["seg_expert"][:ns].cpu().numpy(), [s_[0] for s_ in segs])
        assert np.array_equal(t["seg_row0"][:ns].cpu().numpy(), [s_[1] for s_ in segs])
        assert np.array_equal(t["seg_rows"][:ns].cpu().numpy(), [s_[2] for s_ in segs])
    assert (t["row_expert"][nr:rows_cap].cpu().numpy() == -1).all()  # rows no fat expert fills


def test_e4m3_seg_tables_bit_exact(cuda):
    from mi355moe import e4m3_ext
    g = torch.Generator().manual_seed(3)
    counts = torch.randint(0, 400, (288,), generator=g)          # P ~ 49,000 <= 65,536 rows
    counts[::7] = 0
    P = int(counts.sum())
    se, sr0, sr, ns, nr = e4m3_ext.seg_tables(counts.to(cuda), e4m3_ext.tile_rows(), P)
    local = np.repeat(np.arange(288), counts.numpy())
    o = routing.permutation(local, 288, 1, 1 << 30, e4m3_ext.tile_rows())
    k = int(ns.item())
    assert k == len(o["seg_expert"]) and int(nr.item()) == P
    assert np.array_equal(se[:k].cpu().numpy(), o["seg_expert"])
    assert np.array_equal(sr0[:k].cpu().numpy(), o["seg_row0"])
    assert np.array_equal(sr[:k].cpu().numpy(), o["seg_rows"])


def test_e4m3_seg_tables_refuse_tall_tiles(cuda):
    from mi355moe import _lib, e4m3_ext
    with pytest.raises(_lib.MoeError):
        e4m3_ext.seg_tables(torch.ones(8, dtype=torch.int64, device=cuda), e4m3_ext.tile_rows() + 16, 8)


def _plan_loop(ids, w, n, emap=None):
    """The overlay's plan by plain loops: local ids (map_topk_to_local), rows grouped by local id in pair order with
    the pairs of no local expert (id n) last."""
    T, topk = ids.shape
    flat = ids.reshape(-1)
    local = np.full(flat.size, n, np.int64)
    for j, g_ in enumerate(flat):
        if emap is None:
            local[j] = g_ if 0 <= g_ < n else n
        elif 0 <= g_ < emap.size and 0 <= emap[g_] < n:
            local[j] = emap[g_]
    pos = np.empty(flat.size, np.int64)
    row_token, row_weight, row_expert = [], [], []
    for e in range(n + 1):
        for j in range(flat.size):
            if local[j] == e:
                pos[j] = len(row_token)
                row_token.append(j // topk)
                row_weight.append(w.reshape(-1)[j])
                row_expert.append(e)
    counts = np.array([(local == e).sum() for e in range(n + 1)])
    return local, pos, np.array(row_token), np.array(row_weight, np.float32), np.array(row_expert), counts


@pytest.mark.parametrize("T,topk,use_map", [(5, 8, False), (300, 8, False), (200, 4, True)])
def test_e4m3_plan_vs_loop(cuda, T, topk, use_map):
    from mi355moe import e4m3_ext
    n = 16
    g = np.random.default_rng(T)
    emap = None
    if use_map:                                                       # 24 global ids, 16 local, 8 on other ranks
        emap = np.full(24, -1, np.int64)
        emap[g.permutation(24)[:n]] = np.arange(n)
        ids = np.stack([g.permutation(24)[:topk] for _ in range(T)])
    else:
        ids = np.stack([g.permutation(n)[:topk] for _ in range(T)])
    ids[0, 0] = -1
    ids[T // 2, topk - 1] = 99
    w = g.random((T, topk)).astype(np.float32)
    t = e4m3_ext.plan(torch.from_numpy(ids).to(cuda), torch.from_numpy(w).to(cuda), n,
                      None if emap is None else torch.from_numpy(emap).to(cuda))
    local, pos, rt, rw, re, counts = _plan_loop(ids, w, n, emap)
    assert np.array_equal(t["local"].cpu().numpy(), local)
    assert np.array_equal(t["pos"].cpu().numpy(), pos)
    assert np.array_equal(t["row_token"].cpu().numpy(), rt)
    assert np.array_equal(t["row_weight"].cpu().numpy(), rw)
    assert np.array_equal(t["row_expert"].cpu().numpy(), re)
    assert np.array_equal(t["counts"].cpu().numpy(), counts)
    assert int(t["num_rows"].item()) == int(counts[:n].sum())


def _stored_codes(a8: torch.Tensor) -> np.ndarray:
    """The plain-order codes of rows in the extension's byte order."""
    return e4m3_trellis.from_storage(a8.cpu().numpy())


def _same_codes(got: np.ndarray, ref: np.ndarray) -> bool:
    """e4m3 codes equal byte for byte, except that 0x00 and 0x80 (+0 and -0, one value) count as equal: which exact
    zeros come out negative depends on the operand order inside the butterflies (an all-zero input row gives a mix of
    both on either side)."""
    z = lambda c: np.where(np.asarray(c) == 0x80, 0, np.asarray(c))    # noqa: E731
    return np.array_equal(z(got), z(ref))


@pytest.mark.parametrize("K,xdt", [(1024, torch.bfloat16), (4096, torch.float16)])
def test_e4m3_gathers_write_the_extension_format(cuda, K, xdt):
    """gather2 (per pair, into row pos[j]) and gather_tok (per token): the codes in the extension's byte order and
    the row scales, bit for bit against the oracle's quantiser; rows of skipped pairs stay untouched; out zeroed."""
    from mi355moe import e4m3_ext, synthetic
    n, N, T, topk = 8, 512, 37, 4
    ex = synthetic.exl3_layer(n, K, N, seed=3, device=cuda, uniform_suh=True)
    x = synthetic.activations(T, K, seed=4, device=cuda).to(xdt)
    x[5] = 0                                                         # an all-zero row: scale 1
    ids = synthetic.random_ids(T, n, topk, seed=5, device=cuda)
    ids[2, 1] = -1
    w = synthetic.softmax_weights(T, topk, seed=6, device=cuda)
    t = e4m3_ext.plan(ids, w, n)
    P = T * topk
    a8 = torch.full((P, K), 0xA5, dtype=torch.uint8, device=cuda)
    asc = torch.full((P,), -1.0, device=cuda)
    out = torch.full((T, K), 3.0, device=cuda)
    e4m3_ext.gather2(x, t["local"], t["pos"], ex.tables["gate_suh"], a8, asc, out, topk, n)
    a8t = torch.full((T + 3, K), 0xA5, dtype=torch.uint8, device=cuda)
    asct = torch.full((T + 3,), -1.0, device=cuda)
    e4m3_ext.gather_tok(x, ex.tables["gate_suh"], a8t, asct, None)
    torch.cuda.synchronize()
    assert not out.any()
    x16 = x.to(torch.float16).cpu().numpy()
    suh = ex.w13_suh[0, 0].cpu().numpy()
    codes, sc = e4m3_trellis.act_quant_codes(x16, np.broadcast_to(suh, x16.shape))
    assert _same_codes(_stored_codes(a8t[:T]), codes)
    assert np.array_equal(asct[:T].cpu().numpy(), sc)
    assert (a8t[T:].cpu().numpy() == 0xA5).all() and (asct[T:].cpu().numpy() == -1.0).all()
    pos = t["pos"].cpu().numpy()
    loc = t["local"].cpu().numpy()
    got = _stored_codes(a8)
    for j in range(P):
        if loc[j] >= n:
            assert (a8[pos[j]].cpu().numpy() == 0xA5).all()         # a skipped pair writes nothing
            continue
        assert _same_codes(got[pos[j]], codes[j // topk]) and asc[pos[j]].item() == sc[j // topk]
    assert sc[5] == 1.0 and not (codes[5] & 0x7F).any()            # the zero row: scale 1, zero codes


def _layer_np(ex):
    return _np_layer(ex)


def _down_from_kernel_rows(keep, lay, T, K):
    """The reference's A4 check (code/fork/tests/moee4m3/test_moe_e4m3.py:168-181): the down stage and the weighted
    scatter in float64 from the kernel's own e4m3 down inputs (a8d, dsc) and row tables."""
    nr = int(keep["num_rows"].item())
    re = keep["row_expert"][:nr].cpu().numpy()
    rt = keep["row_token"][:nr].cpu().numpy()
    rw = keep["row_weight"][:nr].cpu().numpy().astype(np.float64)
    qd = e4m3.decode(_stored_codes(keep["a8d"][:nr])).astype(np.float32)
    dsc = keep["dsc"][:nr].cpu().numpy()
    y = np.zeros((T, K), np.float64)
    for e in np.unique(re):
        r = re == e
        yd = e4m3_trellis.down_rows(qd[r], dsc[r], lay["w2_trellis"][e], lay["w2_svh"][e])
        np.add.at(y, rt[r], rw[r, None] * yd)
    return y


def _elementwise_report(got, ref, what):
    bad = ~np.isclose(got, ref, rtol=2e-2, atol=1e-3)
    i = int(np.argmax(np.abs(got - ref) - 2e-2 * np.abs(ref)))
    _say(f"  {what}: {bad.mean():.4%} of elements outside rtol 2e-2 / atol 1e-3; worst got {got.flat[i]:.5f} "
         f"ref {ref.flat[i]:.5f}")
    return float(bad.mean())


@pytest.mark.parametrize("nchunks", [1, 3])
def test_e4m3_chunked_stages_vs_oracle(cuda, nchunks):
    """The chunked schedule (gateup, actq, down per chunk of segments) with each stage checked from the previous
    stage's own output: a16 against the oracle's gate/up of the kernel's e4m3 rows (the reference's A2 bar, rel_l2 <
    2e-4), a8d / dsc bit for bit against the oracle's quantiser of the kernel's a16 (A3), the output against the
    oracle (rel_l2 <= 1e-3) and against fused, whose intermediates are bit-identical."""
    from mi355moe import e4m3_ext, synthetic
    n, K, N, T, topk = 8, 1024, 512, 150, 4
    _say(f"e4m3 chunked stages n={n} K={K} N={N} T={T} nchunks={nchunks}")
    ex = synthetic.calibrated_layer(n, K, N, seed=25, device=cuda)
    x = synthetic.activations(T, K, seed=26, device=cuda)
    ids = synthetic.random_ids(T, n, topk, seed=27, device=cuda)
    ids[3, 2] = -1
    w = synthetic.softmax_weights(T, topk, seed=28, device=cuda)
    keep: dict = {}
    out = e4m3_ext.run(x, ids, w, ex, 10.0, keep=keep, sched={"mode": "chunked", "nchunks": nchunks})
    keep_f: dict = {}
    out_f = e4m3_ext.run(x, ids, w, ex, 10.0, keep=keep_f)
    torch.cuda.synchronize()
    nr = int(keep["num_rows"].item())
    re = keep["row_expert"][:nr].cpu().numpy()
    lay = _layer_np(ex)
    q8 = e4m3.decode(_stored_codes(keep["a8"][:nr])).astype(np.float32)
    asc = keep["asc"][:nr].cpu().numpy()
    a16 = keep["a16"][:nr].cpu().numpy()
    a16_ref = np.empty_like(a16)
    for e in np.unique(re):
        r = re == e
        a16_ref[r] = e4m3_trellis.gateup_rows(q8[r], asc[r], lay["w13_trellis"][e, 0], lay["w13_trellis"][e, 1],
                                              lay["w13_svh"][e, 0], lay["w13_svh"][e, 1], 10.0)
    r16 = _rel(a16, a16_ref)
    _say(f"  A2 a16 rel_l2 {r16:.2e}, {np.mean(a16 == a16_ref):.4%} bit-identical")
    assert r16 < 2e-4
    cd, sd = e4m3_trellis.act_quant_codes(a16, lay["w2_suh"][re])
    assert _same_codes(_stored_codes(keep["a8d"][:nr]), cd)
    assert np.array_equal(keep["dsc"][:nr].cpu().numpy(), sd)
    for k in ("a16", "a8d", "dsc"):
        assert torch.equal(keep[k][:nr], keep_f[k][:nr]), k
    local = routing.map_topk_to_local(ids.cpu().numpy(), n)
    tok, exx, _ = moe.pairs_from_routing(local, w.cpu().numpy(), n, topk)
    ref = e4m3_trellis.forward(lay, x.to(torch.float16).cpu().numpy(), tok, exx, w.cpu().numpy().reshape(-1), 10.0)
    o = out.cpu().numpy().astype(np.float64)
    r = _rel(o, ref)
    _say(f"  output rel_l2 vs oracle {r:.3e}")
    assert r <= 1e-3
    assert _rel(o, out_f.cpu().numpy()) <= 1e-6                      # chunk sums added in another order
    y4 = _down_from_kernel_rows(keep, lay, T, K)
    r4 = _rel(o, y4)
    _say(f"  A4 down from the kernel's a8d: rel_l2 {r4:.2e}")
    assert r4 <= 1e-5 and np.allclose(o, y4, rtol=2e-2, atol=1e-3)
    # end to end the oracle requantises its own a16 (float64 sums): an fp16 ulp on a row's largest element moves
    # that row's scale and re-rounds all its codes, so a few elements leave the elementwise bar (recorded, not held)
    _elementwise_report(o, ref, "end to end vs oracle")


@pytest.mark.parametrize("uniform,out_dtype,down16", [(True, torch.float32, False), (False, torch.float32, False),
                                                      (True, torch.bfloat16, False), (True, torch.float32, True)])
def test_e4m3_ext_run(cuda, uniform, out_dtype, down16):
    """The overlay's default call sequence (plan, then gather_tok when every expert shares one w13 suh, else gather2,
    then fused) against the oracle's e4m3 spec and against the whole-call entry mi355moe_e4m3_moe_forward_ids (same
    kernels; the sums differ only in order). down16: the fp16 down projection (fused variant 16)."""
    from mi355moe import e4m3_ext, ops, synthetic
    n, K, N, T, topk = 8, 1024, 512, 300, 8
    _say(f"e4m3 extension run n={n} K={K} N={N} T={T} uniform_suh={uniform} out={out_dtype} down16={down16}")
    ex = synthetic.calibrated_layer(n, K, N, seed=15, device=cuda, uniform_suh=uniform)
    x = synthetic.activations(T, K, seed=16, device=cuda)
    ids = synthetic.random_ids(T, n, topk, seed=17, device=cuda)
    ids[1, 0] = -1
    w = synthetic.softmax_weights(T, topk, seed=18, device=cuda)
    keep: dict = {}
    sched = {"down16": down16}
    if out_dtype == torch.float32:
        got = e4m3_ext.run(x, ids, w, ex, 10.0, keep=keep, sched=sched)
    else:
        got = torch.full((T, K), 0.5, dtype=torch.bfloat16, device=cuda)     # accumulated into, not zeroed
        e4m3_ext.run(x, ids, w, ex, 10.0, out=got, keep=keep, sched=sched)
    whole = ops.moe_forward_ids_e4m3(ex, x, ids, w, limit=10.0, out_dtype=torch.float32, down16=down16)
    torch.cuda.synchronize()
    assert keep["tok_rows"] == uniform
    local = routing.map_topk_to_local(ids.cpu().numpy(), n)
    tok, exx, _ = moe.pairs_from_routing(local, w.cpu().numpy(), n, topk)
    lay = _np_layer(ex)
    x16 = x.to(torch.float16).cpu().numpy()
    ref = e4m3_trellis.forward(lay, x16, tok, exx, w.cpu().numpy().reshape(-1), 10.0, down16=down16)
    # the gate/up input rows the GEMMs read, as the reference's keep exposes them (a8[row_token[r]] with TOKGATHER)
    nr = int(keep["num_rows"].item())
    rt = keep["row_token"][:nr].cpu().numpy()
    codes, sc = e4m3_trellis.act_quant_codes(x16[rt], lay["w13_suh"][keep["row_expert"][:nr].cpu().numpy(), 0])
    assert _same_codes(_stored_codes(keep["a8"][:nr]), codes)
    assert np.array_equal(keep["asc"][:nr].cpu().numpy(), sc)
    g = got.float().cpu().numpy() - (0.5 if out_dtype == torch.bfloat16 else 0.0)
    r = _rel(g, ref)
    _say(f"  rel_l2 vs oracle {r:.3e}")
    if out_dtype == torch.float32:
        assert r <= 1e-3
        assert _rel(g, whole.cpu().numpy()) <= 1e-5
        if down16:                             # no requantisation: elementwise against the oracle end to end
            assert np.allclose(g, ref, rtol=2e-2, atol=1e-3)
        else:                                  # elementwise from the kernel's own down inputs (A4)
            y4 = _down_from_kernel_rows(keep, lay, T, K)
            assert _rel(g, y4) <= 1e-5 and np.allclose(g, y4, rtol=2e-2, atol=1e-3)
            _elementwise_report(g, ref, "end to end vs oracle")
    else:
        assert r <= 2e-2                       # one bf16 rounding of (0.5 + contribution), steps of 2^-8 .. 2^-7
        assert np.allclose(got.float().cpu().numpy(), 0.5 + ref, rtol=2.0 ** -8, atol=2.0 ** -8)


def test_e4m3_fused_token_rows_of_4_gib(cuda):
    """fused() over token rows whose widened copies pass 4 GiB (tokens x K x 2 bytes; the GEMM's token-row offsets are 32
    bits wide): the rows of the last tokens, bit-equal to the same call over per-row codes."""
    from mi355moe import e4m3_ext, synthetic
    K, N, n, T, rows = 4096, 128, 2, (1 << 19) + 64, 96
    _say(f"e4m3 fused, {T} token rows of {K}")
    ex = synthetic.calibrated_layer(n, K, N, seed=35, device=cuda, uniform_suh=True)
    g = torch.Generator(device=cuda).manual_seed(36)
    tokens = torch.cat([torch.arange(32), torch.arange(T - 64, T)]).to(cuda)   # wrapped, the last 64 would read the first
    tokens = tokens[torch.randperm(rows, generator=g, device=cuda)]
    a8 = torch.zeros(T, K, dtype=torch.uint8, device=cuda)
    asc = torch.zeros(T, device=cuda)
    near = torch.cat([torch.arange(64), torch.arange(T - 64, T)]).to(cuda)
    a8[near] = torch.randint(0, 256, (128, K), generator=g, device=cuda, dtype=torch.int32).to(torch.uint8) & 0xF7
    asc[near] = torch.rand(128, generator=g, device=cuda) * 0.01 + 0.005
    p = ex.tables
    i32 = dict(dtype=torch.int32, device=cuda)
    tabs = (torch.tensor([0, 1], **i32), torch.tensor([0, 61], **i32), torch.tensor([61, 35], **i32),
            torch.tensor([2], **i32))
    rw = torch.rand(rows, generator=g, device=cuda) + 0.1
    out = torch.zeros(T, K, device=cuda)

    def call(codes, scales, variant):
        a16 = torch.empty(rows, N, dtype=torch.float16, device=cuda)
        out.zero_()
        e4m3_ext.fused(codes, scales, None, None, a16, out, p["gate_trellis"], p["up_trellis"], p["gate_svh"],
                       p["up_svh"], p["down_trellis"], p["down_suh"], p["down_svh"], tokens, rw, *tabs, None, 10.0,
                       variant=variant)
        return a16, out[tokens]

    want = call(a8[tokens].contiguous(), asc[tokens].contiguous(), 0)
    got = call(a8, asc, e4m3_ext.TOKEN_ROWS)
    torch.cuda.synchronize()
    assert float(want[0].abs().max()) > 0 and torch.isfinite(want[1]).all()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
