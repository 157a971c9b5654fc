"""Launches whose last work items run in pieces (csrc/split.h).

Each case takes sizes whose plan splits and compares the split call with the same call
without room for its partials (every tile whole): both against the float64 oracle, the split
one no further from it than 1.1x the whole one plus 1e-5 (the pieces are combined in fp32;
what is left is the rounding of P~ against another running maximum). A call must also repeat
bit for bit.
"""
import pytest
import torch

from oracle import attention as orc

pytestmark = pytest.mark.gpu


def _draw(dev, seed, B, H, Lq, Lk, D, dtype):
    g = torch.Generator().manual_seed(seed)

    def r(L, std=1.0):
        return (torch.randn((B, L, H, D), generator=g, dtype=torch.float64) * std).to(dtype).to(dev).transpose(1, 2)

    return r(Lq), r(Lk), r(Lk), r(Lq, 0.1), r(Lk, 0.1), r(Lk, 0.1)


def _no_worse(name, split, whole, ref):
    e, f = orc.rel_l2(split.cpu(), ref), orc.rel_l2(whole.cpu(), ref)
    print(f"  {name} split {e:.2e} whole {f:.2e}", flush=True)
    # fp32: a few more roundings of 2^-24 each
    assert e <= 1.1 * f + (4 * 2 ** -24 if split.dtype == whole.dtype == torch.float32 and f < 1e-5 else 1e-5), (name, e, f)


FWD = [
    # mode, B, H, Lq, Lk, D
    ("jvp", 1, 2, 999, 999, 128),     # 16 tiles alone on the chip
    ("jvp", 1, 2, 999, 2500, 64),
    ("jvp", 1, 1, 130, 545, 128),     # 18 steps, the last one key; a partial query tile
    ("jvp", 2, 1, 257, 2100, 64),
    ("q", 1, 2, 700, 2047, 128),      # key range of the two-workgroups-per-CU kernel
    ("q", 1, 1, 300, 4100, 128),
    ("q", 1, 2, 300, 1000, 64),
    ("plain", 1, 2, 1000, 3100, 128),
    ("plain", 1, 2, 333, 4100, 64),
    ("plain", 1, 1, 1, 3000, 128),    # one query
    ("jvp", 1, 9, 3700, 2500, 128),   # 261 tiles: a full round, then five tiles in pieces
    ("plain", 1, 21, 3200, 3000, 128),  # 525 tiles: a full round of two per CU, then 13
]


FWD_F32 = [
    ("jvp", 1, 2, 256, 256, 64),   # eight steps, a piece each
    ("q", 1, 2, 300, 150, 128),
    ("plain", 1, 1, 100, 2333, 16),
    ("jvp", 1, 1, 129, 1097, 32),
    ("plain", 1, 2, 200, 900, 128),
    ("jvp", 1, 21, 1700, 417, 64),  # 294 tiles: a full round, then 38
]


@pytest.mark.parametrize("mode,B,H,Lq,Lk,D,dtype", [(*c, t) for c in FWD for t in (torch.bfloat16, torch.float16)] +
                         [(*c, torch.float32) for c in FWD_F32])
def test_split_forward(gpu, monkeypatch, mode, B, H, Lq, Lk, D, dtype):
    from dmad_amd import _native as nat
    from dmad_amd.jvp_attention import jvp_attention_forward

    print(f"case split fwd {mode} {B} {H} {Lq} {Lk} {D} {dtype}", flush=True)
    code = nat.dtype_code(dtype)
    nmode = {"plain": nat.DMAD_FWD_PLAIN, "jvp": nat.DMAD_FWD_JVP, "q": nat.DMAD_FWD_JVP_KV_TANGENT_ZERO}[mode]
    q, k, v, tq, tk, tv = _draw(gpu, Lq + Lk + D, B, H, Lq, Lk, D, dtype)
    args = (q, k, v) + ((None,) * 3 if mode == "plain" else (tq, None, None) if mode == "q" else (tq, tk, tv))
    assert nat.fwd_split_bytes(code, nmode, B, H, Lq, Lk, D, D) > 0
    got = jvp_attention_forward(*args, D ** -0.5)
    again = jvp_attention_forward(*args, D ** -0.5)
    monkeypatch.setattr(nat, "fwd_split_bytes", lambda *a: 0)
    whole = jvp_attention_forward(*args, D ** -0.5)
    torch.cuda.synchronize()
    for a, b in zip(got, again):
        assert a is b is None or torch.equal(a, b)
    heads = [0, H - 1] if H > 3 else list(range(H))
    xs = [t[:, heads].cpu().double() for t in (q, k, v, tq, tk if mode == "jvp" else torch.zeros_like(k),
                                               tv if mode == "jvp" else torch.zeros_like(v))]
    ref = orc.jvp_closed_form(*xs)
    for name, a, b, r in zip(("o", "to", "lse", "mu"), got, whole, ref):
        if a is not None:
            _no_worse(name, a[:, heads], b[:, heads], r)


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (128, torch.float16), (64, torch.float32)])
def test_split_forward_with_masked_pieces(gpu, D, dtype):
    """Keys that all score -inf in the last pieces (a -inf feature in K, as a caller's padding
    mask): they weigh nothing, and every row is what the other keys give."""
    from dmad_amd import _native as nat
    from dmad_amd.jvp_attention import jvp_attention_forward

    B, H, Lq, Lk, live = 1, 2, 200, 2000, 700
    assert nat.fwd_split_bytes(nat.dtype_code(dtype), nat.DMAD_FWD_PLAIN, B, H, Lq, Lk, D, D) > 0
    q, k, v, *_ = _draw(gpu, 3, B, H, Lq, Lk, D, dtype)
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    k[:, :, live:, 0] = -float("inf")
    o, _, lse, _ = jvp_attention_forward(q, k, v, None, None, None, D ** -0.5)
    ro, rlse = orc.math_attention(q.cpu().double(), k[:, :, :live].cpu().double(), v[:, :, :live].cpu().double(), D ** -0.5)
    assert orc.rel_l2(o.cpu(), ro) <= 1e-2
    assert float((lse.cpu().double() - rlse).abs().max()) <= 2e-3


@pytest.mark.parametrize("mode", ["jvp", "q"])
@pytest.mark.parametrize("Lk,live,D,dtype", [(2000, 700, 64, torch.bfloat16), (2000, 700, 128, torch.bfloat16),
                                             (900, 300, 64, torch.float32)])
def test_split_jvp_with_masked_pieces(gpu, mode, Lk, live, D, dtype):
    """The same with tangents: scores that overflow to -inf, as a caller's finite mask feature can
    (an infinite one has no finite tangent)."""
    from dmad_amd import _native as nat
    from dmad_amd.jvp_attention import jvp_attention_forward

    print(f"case masked jvp pieces {mode} {Lk} {D} {dtype}", flush=True)
    assert nat.fwd_split_bytes(nat.dtype_code(dtype), nat.DMAD_FWD_JVP, 1, 2, 200, Lk, D, D) > 0
    q, k, v, tq, tk, tv = _draw(gpu, 3, 1, 2, 200, Lk, D, dtype)
    for t in (k, tq, tk):
        t[..., 0] = 0.0
    q[..., 0] = 1e20
    k[:, :, live:, 0] = -1e30
    if mode == "q":
        tk, tv = torch.zeros_like(k), torch.zeros_like(v)
    got = jvp_attention_forward(q, k, v, tq, *((tk, tv) if mode == "jvp" else (None, None)), D ** -0.5)
    ref = orc.jvp_closed_form(*(t.cpu().double()[:, :, :live] if t.shape[2] == Lk else t.cpu().double()
                                for t in (q, k, v, tq, tk, tv)))
    for name, a, r in zip(("o", "to", "lse", "mu"), got, ref):
        assert orc.rel_l2(a.cpu(), r) <= (1e-2 if dtype == torch.bfloat16 else 1e-5), name


@pytest.mark.parametrize("mode", ["plain", "jvp"])
@pytest.mark.parametrize("offset", [-2.0 ** 30, 2.0 ** 17])
@pytest.mark.parametrize("Lk,D,dtype", [(2010, 64, torch.bfloat16), (2010, 128, torch.bfloat16), (900, 64, torch.float32)])
def test_split_forward_beside_a_large_common_score(gpu, mode, offset, Lk, D, dtype):
    """Rows all of whose scores are one large value (a caller's mask as a feature of K, in rows that
    it masks throughout): a piece weighs by the number of its keys, which differ."""
    from dmad_amd import _native as nat
    from dmad_amd.jvp_attention import jvp_attention_forward

    print(f"case common score {mode} {offset} {Lk} {D} {dtype}", flush=True)
    nmode = nat.DMAD_FWD_PLAIN if mode == "plain" else nat.DMAD_FWD_JVP
    assert nat.fwd_split_bytes(nat.dtype_code(dtype), nmode, 1, 2, 200, Lk, D, D) > 0
    q, k, v, tq, tk, tv = _draw(gpu, 5, 1, 2, 200, Lk, D, dtype)
    v += (torch.arange(Lk, device=gpu) / Lk).to(dtype)[None, None, :, None]  # uneven over the keys
    q.zero_()
    q[..., 0] = 1.0
    tq[..., 0] = 0.0
    k[..., 0] = 0.0
    xs = (q, k, v, tq, tk, tv)
    ref = orc.jvp_closed_form(*(t.cpu().double() for t in xs), sm_scale=1.0)  # a common score changes nothing
    k[..., 0] = offset
    o, to, _, mu = jvp_attention_forward(*(xs if mode == "jvp" else (q, k, v, None, None, None)), 1.0)
    assert orc.rel_l2(o.cpu(), ref[0]) <= (1e-2 if dtype == torch.bfloat16 else 1e-5)
    if mode == "jvp":
        assert orc.rel_l2(to.cpu(), ref[1]) <= 1e-2 and orc.rel_l2(mu.cpu(), ref[3]) <= 1e-2


@pytest.mark.parametrize("mode", ["plain", "jvp"])
@pytest.mark.parametrize("B,H,Lq,Lk,D,dtype", [
    (1, 2, 200, 2000, 64, torch.bfloat16), (1, 2, 200, 2000, 128, torch.bfloat16), (1, 2, 200, 900, 64, torch.float32),
    (1, 21, 3200, 3000, 128, torch.bfloat16)])  # the last one: full rounds of whole tiles, too
@pytest.mark.parametrize("whole", [False, True])
def test_split_forward_at_the_lowest_scores(gpu, monkeypatch, whole, mode, B, H, Lq, Lk, D, dtype):
    """Rows all of whose scores are bf16's lowest value (a caller's mask as a feature of K): equal
    scores, finite ones, so the softmax is uniform, as in a launch that does not split."""
    from dmad_amd import _native as nat
    from dmad_amd.jvp_attention import jvp_attention_forward

    print(f"case lowest scores {mode} {B} {H} {Lq} {Lk} {D} {dtype}", flush=True)
    nmode = nat.DMAD_FWD_PLAIN if mode == "plain" else nat.DMAD_FWD_JVP
    assert nat.fwd_split_bytes(nat.dtype_code(dtype), nmode, B, H, Lq, Lk, D, D) > 0
    q, k, v, tq, tk, tv = _draw(gpu, 5, B, H, Lq, Lk, D, dtype)
    if whole:
        monkeypatch.setattr(nat, "fwd_split_bytes", lambda *a: 0)
    q.zero_()
    q[..., 0] = 1.0
    k[..., 0] = torch.finfo(torch.bfloat16).min
    tq[..., 0] = 0.0
    scale = 0.6931471824645996  # times log2(e) rounds to 1: the scores in the log2 domain are as given
    xs = (q, k, v, tq, tk, tv) if mode == "jvp" else (q, k, v, None, None, None)
    o, to, lse, mu = (None if t is None else t[:, -1:].cpu() for t in jvp_attention_forward(*xs, scale))
    assert bool((lse == torch.finfo(torch.bfloat16).min * 0.6931471805599453).all())
    k[..., 0] = 0.0  # equal scores for the oracle (exp(S - LSE) in float64 would lose log(Lk) beside 1e38)
    ref = orc.jvp_closed_form(*(t[:, -1:].cpu().double() for t in (q, k, v, tq, tk, tv)), sm_scale=scale)
    assert orc.rel_l2(o, ref[0]) <= 1e-2
    if mode == "jvp":
        assert orc.rel_l2(to, ref[1]) <= 1e-2 and orc.rel_l2(mu, ref[3]) <= 1e-2


BWD = [
    # B, H, Lq, Lk, D, full derivative with tangent gradients
    (1, 2, 2300, 2300, 64, False),
    (1, 2, 999, 999, 128, False),    # recomputing query pass
    (1, 2, 2111, 2111, 128, False),  # stored score gradients
    (1, 2, 700, 905, 128, True),
    (1, 2, 2500, 2500, 64, True),    # the tangent passes of 64-wide heads
    (2, 1, 130, 3000, 128, False),   # few query tiles, a partial one
    (1, 1, 3000, 33, 64, False),     # one key tile, 94 query steps
    (1, 9, 3700, 3700, 128, False),  # 261 key tiles: one after the full round, in pieces
    (1, 9, 3700, 3700, 128, True),
    (1, 27, 2500, 2500, 64, False),  # 540 key tiles of two per CU; 540 query tiles of three
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Lq,Lk,D,full", BWD)
def test_split_backward(gpu, monkeypatch, B, H, Lq, Lk, D, full, dtype):
    """The tiles' P and dS do not change, only the order in which fp32 sums add up, so a split
    gradient differs from the whole one by output roundings that fall the other way."""
    from dmad_amd import _native as nat
    from dmad_amd.jvp_attention import jvp_attention_backward, jvp_attention_forward

    print(f"case split bwd {B} {H} {Lq} {Lk} {D} full={full} {dtype}", flush=True)
    code = nat.dtype_code(dtype)
    assert nat.bwd_split_bytes(code, full, full, B, H, Lq, Lk, D) > 0
    q, k, v, tq, tk, tv = _draw(gpu, Lq + Lk + D, B, H, Lq, Lk, D, dtype)
    do, _, _, dto, _, _ = _draw(gpu, 1, B, H, Lq, Lk, D, dtype)
    s = D ** -0.5
    o, to, lse, mu = jvp_attention_forward(q, k, v, tq, tk, tv, s)

    def backward():
        return jvp_attention_backward(q, k, v, tq, tk, tv, o, to, lse, mu, do, dto if full else None, s, full)

    got, again = backward(), backward()
    monkeypatch.setattr(nat, "bwd_split_bytes", lambda *a: 0)
    whole = backward()
    torch.cuda.synchronize()
    names = ("dq", "dk", "dv", "dtq", "dtk", "dtv")
    for name, a, b, w in zip(names, got, again, whole):
        assert a is b is w is None or (torch.equal(a, b) and
                                       orc.rel_l2(a.cpu(), w.cpu()) <= (2 ** -9 if dtype == torch.bfloat16 else 2 ** -12)), name
    if H > 2:
        return
    xs = [t.cpu().double() for t in (q, k, v, tq, tk, tv, do, dto)]
    ref = orc.grads_full(*xs) if full else orc.grads_dout_only(*xs[:3], xs[6])
    for name, a, w, r in zip(names, got, whole, ref):
        _no_worse(name, a, w, r)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("kv_tangents", [True, False])
@pytest.mark.parametrize("hint", [60, 3000])  # a few pieces per task; more pieces than some tasks have tiles
def test_split_block_sparse_forward(gpu, hint, kv_tangents, D, dtype):
    """Tasks of unequal lengths, ranges off the tile grid, a group without keys and rows that no
    task covers: split (the mask's length hint set by hand) against whole and the oracle."""
    import dataclasses

    from dmad_amd import _native as nat
    from dmad_amd import magimask as mm
    from dmad_amd.jvp_attention import jvp_attention_forward_magi
    from oracle import magi as om

    print(f"case split magi hint={hint} kv={kv_tangents} D={D} {dtype}", flush=True)
    B, H, Lq, Lk = 1, 2, 700, 1300
    groups = [(0, 200, [(0, 40)]), (200, 330, [(33, 500), (777, 1300)]), (330, 400, []), (400, 650, [(5, 1290)])]
    keys = [r for g in groups for r in g[2]]
    first = [sum(len(g[2]) for g in groups[:i]) for i in range(len(groups) + 1)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)  # noqa: E731
    qu = i32([[g[0], g[1]] for g in groups])
    tg, tq_ = mm.build_qtile_tasks(qu, Lq, 128)
    mask = mm.MagiMask(qu, i32(keys), i32(first), tg, tq_, len(groups), int(tg.numel()), 128)
    code = nat.dtype_code(dtype)
    split = dataclasses.replace(mask, key_tiles=hint)
    assert nat.magi_split_bytes(code, mask.T, hint, B, H, D, D) > 0
    q, k, v, tq, tk, tv = _draw(gpu, D, B, H, Lq, Lk, D, dtype)
    tk, tv = (tk, tv) if kv_tangents else (None, None)
    whole = jvp_attention_forward_magi(q, k, v, tq, tk, tv, D ** -0.5, mask)
    got = jvp_attention_forward_magi(q, k, v, tq, tk, tv, D ** -0.5, split)
    again = jvp_attention_forward_magi(q, k, v, tq, tk, tv, D ** -0.5, split)
    torch.cuda.synchronize()
    allow = torch.zeros(Lq, Lk, dtype=torch.bool)
    for a, b, rs in groups:
        for s, e in rs:
            allow[a:b, s:e] = True
    xs = [t.cpu() for t in (q, k, v, tq)] + [(t if t is not None else torch.zeros_like(k)).cpu() for t in (tk, tv)]
    ref = om.masked_jvp(*xs, allow, D ** -0.5)
    for name, a, b, w, r in zip(("o", "to", "lse", "mu"), got, again, whole, ref):
        assert torch.equal(a[:, :, :650], b[:, :, :650]), name  # rows from 650 on are nobody's
        keep = torch.cat([torch.arange(330), torch.arange(400, 650)])
        _no_worse(name, a[:, :, keep], w[:, :, keep], r[:, :, keep])
        assert torch.equal(a[:, :, 330:400], w[:, :, 330:400]), name  # no keys: zeros, LSE -inf


@pytest.mark.parametrize("B,H,D,dtype", [(1, 2, 128, torch.bfloat16), (3, 1, 128, torch.float16), (1, 3, 64, torch.bfloat16),
                                         (2, 1, 64, torch.float16)])
@pytest.mark.parametrize("kv_tangents", [True, False])
def test_split_block_sparse_forward_after_full_rounds(gpu, kv_tangents, B, H, D, dtype):
    """Masks of more tasks than one round takes, up to three heads: whole tasks first, dealt over the
    chip from the last one down, then the rest in pieces."""
    import dataclasses

    from dmad_amd import _native as nat
    from dmad_amd import magimask as mm
    from dmad_amd.jvp_attention import jvp_attention_forward_magi
    from oracle import magi as om

    slots = 256 if D == 128 else 512  # workgroups of a round
    groups, Lk = 8, 1700 if D == 128 else 3300
    tiles = (slots + slots // 16) // (B * H) + 1  # query tiles of a head: a round and a few
    Lq = 128 * tiles - 60
    edges = [Lq * i // groups + 17 * (0 < i < groups) for i in range(groups + 1)]
    rects = [(a, b, 0, Lk * (i + 1) // groups) for i, (a, b) in enumerate(zip(edges, edges[1:]))]
    rects += [(a, b, Lk - 40 * (i + 1), Lk - 5) for i, (a, b) in enumerate(zip(edges, edges[1:]))]
    qr, kr = (torch.tensor([x[j:j + 2] for x in rects], dtype=torch.int32, device=gpu) for j in (0, 2))
    mask = mm.prepare_magi_csr_and_tasks(qr, kr, Q_real=Lq, KV_real=Lk)
    print(f"case split magi rounds B={B} H={H} D={D} kv={kv_tangents} {dtype}: {mask.T * B * H} tasks", flush=True)
    code = nat.dtype_code(dtype)
    assert mask.T * B * H > slots and nat.magi_split_bytes(code, mask.T, mask.key_tiles, B, H, D, D) > 0
    q, k, v, tq, tk, tv = _draw(gpu, D, B, H, Lq, Lk, D, dtype)
    tk, tv = (tk, tv) if kv_tangents else (None, None)
    got, again = (jvp_attention_forward_magi(q, k, v, tq, tk, tv, D ** -0.5, mask) for _ in range(2))
    whole = jvp_attention_forward_magi(q, k, v, tq, tk, tv, D ** -0.5, dataclasses.replace(mask, key_tiles=0))
    torch.cuda.synchronize()
    # every row against the launch that does not split (P~ rounded against another maximum: at most
    # both errors, 2.4e-3 in bf16 and 3e-4 in fp16 each), and some rows of every group, in the first
    # and the last head, against the oracle
    rows = torch.cat([torch.arange(a, b, 61) for a, b in zip(edges, edges[1:])])
    allow = torch.zeros(len(rows), Lk, dtype=torch.bool)
    for a, b, s, e in rects:
        allow[(rows >= a) & (rows < b), s:e] = True
    zeros = torch.zeros_like(k)
    for b, h in ((0, 0), (B - 1, H - 1)):
        xs = [(zeros if t is None else t)[b:b + 1, h:h + 1].cpu() for t in (q, k, v, tq, tk, tv)]
        xs[0], xs[3] = xs[0][:, :, rows], xs[3][:, :, rows]
        ref = om.masked_jvp(*xs, allow, D ** -0.5)
        for name, a, w, r in zip(("o", "to", "lse", "mu"), got, whole, ref):
            _no_worse(name, a[b:b + 1, h:h + 1, rows], w[b:b + 1, h:h + 1, rows], r)
    for name, a, c, w in zip(("o", "to", "lse", "mu"), got, again, whole):
        assert torch.equal(a, c), name
        for b in range(B):
            for h in range(H):
                assert orc.rel_l2(a[b, h].cpu(), w[b, h].cpu()) <= (6e-3 if dtype == torch.bfloat16 else 1e-3), (name, b, h)
