"""Prompt attention of two tiles a wavefront with masks, sinks, gates and float output, against a plain computation in double:
head sizes and groups, windows and chunks that cut inside a 32-key chunk and across a wavefront's tokens, histories in the
cache; which calls take it (GPU)."""
import math
from types import SimpleNamespace

import pytest
import torch

from test_wide_attention_gpu import element_order

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SPANS = [(0, 131), (70, 96), (5, 6), (33, 64), (200, 203), (0, 99)]         # (first new token, length) of every sequence


def cached(spans, heads, hd, page, g, keys, odd=()):
    """A shuffled page table, the pool, and every sequence's rows."""
    width = max(-(-b // page) for _, b in spans)
    place = torch.randperm(width * len(spans), generator=torch.Generator().manual_seed(3)).view(len(spans), width)
    pool, rows = torch.zeros(width * len(spans), page * heads * hd, dtype=torch.bfloat16), []
    for s, (_, b) in enumerate(spans):
        x = torch.randn(b, heads, hd, generator=g).to(torch.bfloat16)
        for t, f, value in odd:
            if t < b:
                x[t, t % heads, f % hd] = value
        flat = torch.zeros(width * page * heads * hd, dtype=torch.bfloat16)
        flat[element_order(b, heads, hd, keys).flatten()] = x.flatten()
        pool[place[s]] = flat.view(width, -1)
        rows.append(x.double())
    return place.int().to(DEV), pool.view(-1, page, heads * hd).to(DEV), rows


def tokens(spans):
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    return i32([t for a, b in spans for t in range(a, b)]), i32([s for s, (a, b) in enumerate(spans) for _ in range(a, b)])


def expected(q, k, v, p, scale, opt, sink, gate):
    """(result, sum of the absolute terms) of a token at position p: [heads, hd]."""
    j, chunk, window = torch.arange(p + 1), opt.get("chunk", 0), opt.get("window", 0)
    sees = (j // chunk == p // chunk) if chunk else (p - j < window) if window else torch.ones(p + 1, dtype=torch.bool)
    sc = torch.einsum("hd,jhd->hj", q, k[:p + 1][sees]) * scale
    if sink is not None:
        sc = torch.cat([sc, sink.double()[:, None]], 1)
    terms = torch.softmax(sc, -1)[:, :int(sees.sum()), None] * v[:p + 1][sees].transpose(0, 1)
    want, size = terms.sum(1), terms.abs().sum(1)
    return (want, size) if gate is None else (want * torch.sigmoid(gate.double()), size * torch.sigmoid(gate.double()))


@pytest.mark.parametrize("waves", [1, 2, 4])
@pytest.mark.parametrize("nh,nkv,hd,opt", [
    (32, 8, 128, {}), (32, 8, 128, {"window": 37, "sink": True}), (4, 4, 64, {"chunk": 48, "gate": True}), (6, 2, 80, {"window": 1}),
    (16, 1, 16, {"window": 100, "out": torch.float32, "gate": True}), (20, 1, 48, {"chunk": 7, "sink": True, "page": 96}),
    (8, 1, 128, {"chunk": 64, "out": torch.float32, "odd": True}), (32, 8, 32, {"window": 64, "odd": True}), (8, 8, 64, {"odd": True}),
])
def test_prompts_with_masks_sinks_and_gates(nh, nkv, hd, opt, waves):
    from cpmcu_amd import ops
    page, g = opt.get("page", 64), torch.Generator().manual_seed(nh + hd)
    odd = [(37, 5, math.inf), (38, 5, -math.inf), (90, 1, math.nan), (91, 3, -math.inf), (130, 0, math.inf)] if opt.get("odd") else []
    table, kpool, ks = cached(SPANS, nkv, hd, page, g, True)
    _, vpool, vs = cached(SPANS, nkv, hd, page, g, False, odd)
    pos, slot = tokens(SPANS)
    n, scale, rep = pos.numel(), 1.3 * hd ** -0.5, nh // nkv
    q = torch.randn(n, nh, hd, generator=g).to(torch.bfloat16)
    sink = torch.randn(nh, generator=g) if opt.get("sink") else None
    gate = torch.randn(n, nh * hd, generator=g).to(torch.bfloat16) if opt.get("gate") else None
    dev = lambda t: None if t is None else t.to(DEV)
    out = torch.full((n, nh * hd), 7.0, dtype=opt.get("out", torch.bfloat16), device=DEV)
    tiles = ops.prefill_tiles([b - a for a, b in SPANS], ops.attention_prefill_tokens_per_wave(nh, nkv, 2), DEV)
    ops.attention_prefill_mfma(dev(q.view(n, -1)), out, tiles, nh, nkv, hd, scale, kpool, vpool, table, page, pos, slot, 2, waves,
                               opt.get("chunk", 0), opt.get("window", 0), dev(sink), dev(gate), True)
    got = out.double().cpu().view(n, nh, hd)
    other = torch.empty_like(out)
    tpt = ops.attention_general_tokens_per_tile(n, nh, nkv, hd)
    ops.attention_general_mfma(dev(q.view(n, -1)), other, nh, nkv, hd, hd, scale, kpool, vpool, table, page, pos, slot, opt.get("chunk", 0),
                               tiles=ops.prefill_tiles([b - a for a, b in SPANS], tpt, DEV) if tpt > 1 else None, tokens_per_tile=tpt,
                               window=opt.get("window", 0), sink=dev(sink), gate=dev(gate))
    # one wavefront a group of tiles: the general kernel's results; infinities and NaNs among the values reach the tokens that
    # they reach there, whose tiles visit the same chunks of keys, and no other
    if waves == 1 and 16 % rep == 0:
        assert torch.equal(out.nan_to_num(7.0), other.nan_to_num(7.0))
    fine = torch.isfinite(other.cpu()).view(n, nh, hd)
    assert torch.equal(torch.isfinite(got), fine) and bool(fine.all()) == (not odd) and bool(fine[:30].all())
    for t, (p, s) in enumerate(zip(pos.tolist(), slot.tolist())):
        want, size = expected(q[t].double(), ks[s].repeat_interleave(rep, 1), vs[s].repeat_interleave(rep, 1), p, scale, opt, sink,
                              None if gate is None else gate[t].view(nh, hd))
        # weights rounded to bf16 (half an ulp each) against values of that size, and the output's own rounding
        assert bool(((got[t] - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-5)[fine[t]].all()), (t, p, s)


@pytest.mark.parametrize("waves", [1, 2, 4])
@pytest.mark.parametrize("nh,nkv,hd,opt", [
    (32, 8, 128, {}), (4, 4, 64, {"window": 37}), (8, 2, 80, {"chunk": 48, "sink": True, "gate": True}), (16, 1, 32, {"window": 70, "out": torch.float32}),
])
def test_infinities_and_nans_in_queries_and_keys(nh, nkv, hd, opt, waves):
    """Scores that are infinite or no numbers: the general kernel's results (with one wavefront a group to the last bit), and
    rows that see none of them beside rows that do."""
    from cpmcu_amd import ops
    page, g = 64, torch.Generator().manual_seed(nh + hd)
    odd = [(37, 5, math.inf), (60, 2, -math.inf), (90, 1, math.nan), (130, 0, math.inf), (64, 3, -math.nan)]
    table, kpool, _ = cached(SPANS, nkv, hd, page, g, True, odd)
    _, vpool, _ = cached(SPANS, nkv, hd, page, g, False)
    pos, slot = tokens(SPANS)
    n, scale = pos.numel(), 1.3 * hd ** -0.5
    q = torch.randn(n, nh, hd, generator=g).to(torch.bfloat16)
    for t, value in ((3, math.nan), (17, math.inf), (18, -math.inf), (n - 2, math.nan), (n - 60, math.inf)):
        q[t, t % nh, t % hd] = value
    q[25, :, 1] = math.inf
    sink = torch.randn(nh, generator=g) if opt.get("sink") else None
    gate = torch.randn(n, nh * hd, generator=g).to(torch.bfloat16) if opt.get("gate") else None
    dev = lambda t: None if t is None else t.to(DEV)
    out, other = (torch.full((n, nh * hd), 7.0, dtype=opt.get("out", torch.bfloat16), device=DEV) for _ in range(2))
    rows, shape = dev(q.view(n, -1)), (scale, kpool, vpool, table, page, pos, slot)
    tiles = ops.prefill_tiles([b - a for a, b in SPANS], ops.attention_prefill_tokens_per_wave(nh, nkv, 2), DEV)
    ops.attention_prefill_mfma(rows, out, tiles, nh, nkv, hd, *shape, 2, waves, opt.get("chunk", 0), opt.get("window", 0), dev(sink), dev(gate), True)
    tpt = ops.attention_general_tokens_per_tile(n, nh, nkv, hd)
    ops.attention_general_mfma(rows, other, nh, nkv, hd, hd, *shape, opt.get("chunk", 0),
                               tiles=ops.prefill_tiles([b - a for a, b in SPANS], tpt, DEV) if tpt > 1 else None, tokens_per_tile=tpt,
                               window=opt.get("window", 0), sink=dev(sink), gate=dev(gate))
    assert torch.equal(out.isnan(), other.isnan()) and torch.equal(out.isinf(), other.isinf())
    assert bool(out.isnan().any()) and bool(out.isfinite().any())
    if waves == 1:
        assert torch.equal(out.nan_to_num(7.0), other.nan_to_num(7.0))
    else:       # another order of the same sums: weights of half an ulp and the output's rounding, values of about 4 at most
        fine = other.isfinite()
        assert float((out - other)[fine].abs().max()) <= 2.0 ** -8 * 8


@pytest.mark.parametrize("spread", [1.0, 3.0])
def test_weights_round_no_worse_than_in_the_general_kernel(spread):
    from cpmcu_amd import ops
    L, nh, nkv, hd, page = 512, 16, 4, 128, 64
    g = torch.Generator().manual_seed(int(spread))
    table, kpool, ks = cached([(0, L)], nkv, hd, page, g, True)
    _, vpool, vs = cached([(0, L)], nkv, hd, page, g, False)
    pos, slot = tokens([(0, L)])
    q = (spread * torch.randn(L, nh, hd, generator=g)).to(torch.bfloat16)
    rows, shape = q.view(L, -1).to(DEV), (hd ** -0.5, kpool, vpool, table, page, pos, slot)
    outs = [torch.empty(L, nh * hd, device=DEV) for _ in range(4)]
    tiles = ops.prefill_tiles([L], ops.attention_prefill_tokens_per_wave(nh, nkv, 2), DEV)
    for waves, out in zip((1, 2, 4), outs):
        ops.attention_prefill_mfma(rows, out, tiles, nh, nkv, hd, *shape, 2, waves, general=True)
    ops.attention_general_mfma(rows, outs[3], nh, nkv, hd, hd, *shape)
    k, v = (x[0].repeat_interleave(nh // nkv, 1) for x in (ks, vs))
    s = torch.einsum("thd,jhd->htj", q.double(), k) * hd ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    want = torch.einsum("htj,jhd->thd", torch.softmax(s, -1), v).reshape(L, -1)
    off = [float((x.double().cpu() - want).norm()) for x in outs]
    assert max(off[:3]) <= 1.05 * off[3], off                       # 5% for other orders of summing


@pytest.mark.parametrize("change,taken", [
    ({}, "prefill"), ({"window": 96, "keep_first": 3}, "prefill"), ({"window": 95, "keep_first": 3}, "general"), ({"window": 95}, "prefill"),
    ({"chunk": 40, "sink": True}, "prefill"), ({"softcap": 3.0}, "general"), ({"hdv": 112}, "general"), ({"v_share": 2}, "general"),
    ({"out": torch.bfloat16}, "attention"), ({"few": True}, "general"),
])
def test_which_prompts_take_the_kernel(change, taken, monkeypatch):
    """(positions up to 95: a window of 96 cuts nothing off, one of 95 does; up to 256 tokens stay with the general kernel)"""
    from cpmcu_amd import ops
    nh, nkv, hd, hdv, page, spans = 8, 4, 64, change.get("hdv", 64), 64, [(0, 80)] * 3 + [(80 if change.get("few") else 79, 96)]
    nvh, g = nkv // change.get("v_share", 1), torch.Generator().manual_seed(1)
    table, kpool, ks = cached(spans, nkv, hd, page, g, True)
    _, vpool, vs = cached(spans, nvh, hdv, page, g, False)
    pos, slot = tokens(spans)
    ctx = SimpleNamespace(single_token=False, max_pos=95, q_lens=[b - a for a, b in spans], extras={}, positions=pos, tok_slot=slot)
    n = pos.numel()
    q, out = torch.randn(n, nh, hd, generator=g).to(torch.bfloat16), torch.empty(n, nh * hdv, dtype=change.get("out", torch.float32), device=DEV)
    sink = torch.randn(nh, generator=g) if change.get("sink") else None
    called = []
    for name in ("attention_prefill_mfma", "attention_general_mfma"):
        monkeypatch.setattr(ops, name, lambda *a, _f=getattr(ops, name), _n=name, **k: (called.append(_n + "+" * bool(k.get("general"))), _f(*a, **k)))
    kw = {k: change[k] for k in ("window", "keep_first", "chunk", "v_share") if k in change}
    ops.attention_any(q.view(n, -1).to(DEV), out, nh, nkv, hd, hdv, hd ** -0.5, kpool, vpool, table, page, ctx,
                      sink=None if sink is None else sink.to(DEV), softcap=change.get("softcap", 0.0), **kw)
    assert called == [{"prefill": "attention_prefill_mfma+", "general": "attention_general_mfma", "attention": "attention_prefill_mfma"}[taken]]
    if "softcap" in change or "keep_first" in change:
        return
    for t, (p, s) in enumerate(zip(pos.tolist(), slot.tolist())):
        want, size = expected(q[t].double(), ks[s].repeat_interleave(nh // nkv, 1), vs[s].repeat_interleave(nh // nvh, 1), p, hd ** -0.5, change, sink, None)
        assert bool(((out[t].double().cpu().view(nh, hdv) - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-5).all()), (t, p, s)
