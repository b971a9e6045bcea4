"""Prompt attention with wide values against a plain computation in double: heads a group, key and value sizes at and beside
the built ones, masks, sinks, caps, gates, shared values, page sizes, tiles that end early, a history in the cache (GPU)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def element_order(tokens, heads, hd, keys):
    """Where element [token, head, feature] of a run of pages lies (pages one behind the other)."""
    t, h, d = torch.arange(tokens)[:, None, None], torch.arange(heads)[None, :, None], torch.arange(hd)[None, None]
    base, i = ((t // 32) * heads + h) * 32 * hd, t % 32
    if keys:
        return base + ((i // 4) % 2) * hd * 16 + ((i // 8) * 4 + i % 4) * 8 + (d // 8) * 128 + d % 8
    return base + (i // 8) * 128 + i % 8 + (d // 16) * 512 + (d % 16) * 8


CASES = [
    # heads, kv heads, key features, cached as, value features, v_share, options
    (32, 1, 576, 576, 512, 1, {}),
    (32, 1, 576, 576, 512, 1, {"window": 37, "sink": True, "gate": True}),
    (32, 8, 128, 128, 256, 2, {"out": torch.float32}),
    (4, 4, 120, 128, 144, 1, {"chunk": 48}),
    (64, 1, 192, 192, 512, 1, {"softcap": 3.0}),
    (6, 3, 64, 64, 260, 3, {"window": 20, "keep_first": 5, "page": 32}),
    (16, 2, 320, 320, 132, 1, {"page": 96, "sink": True}),
]


@pytest.mark.parametrize("nh,nkv,hdk,pool_hdk,hdv,v_share,opt", CASES)
def test_wide_prompt_attention(nh, nkv, hdk, pool_hdk, hdv, v_share, opt):
    from cpmcu_amd import ops
    page, pool_hdv, nvh = opt.get("page", 64), -(-hdv // 16) * 16, nkv // v_share
    g = torch.Generator().manual_seed(hdk + hdv)
    spans = [(0, 131), (70, 96), (5, 6), (33, 64)]                 # (first new token, length) of every sequence
    pages = [-(-b // page) for _, b in spans]
    place = torch.randperm(sum(pages), generator=g)
    table = torch.zeros(len(spans), max(pages), dtype=torch.int32)
    kpool = torch.zeros(sum(pages), page, nkv * pool_hdk, dtype=torch.bfloat16)
    vpool = torch.zeros(sum(pages), page, nvh * pool_hdv, dtype=torch.bfloat16)
    ks, vs, at = [], [], 0
    for s, (_, length) in enumerate(spans):
        k = torch.randn(length, nkv, hdk, generator=g).to(torch.bfloat16)
        v = torch.randn(length, nvh, hdv, generator=g).to(torch.bfloat16)
        ks.append(k.double())
        vs.append(v.double())
        mine = place[at:at + pages[s]]
        at += pages[s]
        table[s, :pages[s]] = mine.int()
        for pool, x, heads, hd, is_key in ((kpool, k, nkv, pool_hdk, True), (vpool, v, nvh, pool_hdv, False)):
            flat = torch.zeros(pages[s] * page * heads * hd, dtype=torch.bfloat16)
            order = element_order(length, heads, hd, is_key)[..., :x.shape[-1]]
            flat[order.flatten()] = x.flatten()
            pool[mine] = flat.view(pages[s], page, heads * hd)
    pos = torch.cat([torch.arange(a, b) for a, b in spans]).int()
    slot = torch.cat([torch.full((b - a,), s) for s, (a, b) in enumerate(spans)]).int()
    n = pos.numel()
    q = torch.randn(n, nh, hdk, generator=g).to(torch.bfloat16)
    sink = torch.randn(nh, generator=g) if opt.get("sink") else None
    gate = torch.randn(n, nh * hdv, generator=g).to(torch.bfloat16) if opt.get("gate") else None
    scale, cap = 1.3 * hdk ** -0.5, opt.get("softcap", 0.0)
    chunk, window, keep = opt.get("chunk", 0), opt.get("window", 0), opt.get("keep_first", 0)
    dev = lambda t: None if t is None else t.to(DEV)
    tiles = ops.prefill_tiles([b - a for a, b in spans], 64 * nkv // nh, DEV)
    out = torch.full((n, nh * hdv), float("nan"), dtype=opt.get("out", torch.bfloat16), device=DEV)
    assert ops.attention_wide_prefill_ok(dev(q), nh, nkv, hdk, hdv, pool_hdk, pool_hdv, page)
    ops.attention_wide_prefill(dev(q.view(n, -1)), out, tiles, nh, nkv, hdk, hdv, scale, dev(kpool), dev(vpool), dev(table), page,
                               dev(pos), dev(slot), chunk, window, keep, dev(sink), v_share, dev(gate), cap)
    got = out.double().cpu().view(n, nh, hdv)
    rep = nh // nkv
    for t in range(n):
        p, s = int(pos[t]), int(slot[t])
        k, v = ks[s][:p + 1].repeat_interleave(rep, 1), vs[s][:p + 1].repeat_interleave(rep * v_share, 1)
        sc = torch.einsum("hd,jhd->hj", q[t].double(), k) * scale
        sc = cap * torch.tanh(sc / cap) if cap else sc
        j = torch.arange(p + 1)
        hidden = (j // chunk != p // chunk) if chunk else ((p - j >= window) & (j >= keep)) if window else torch.zeros(p + 1, dtype=torch.bool)
        sc = sc.masked_fill(hidden, -math.inf)
        if sink is not None:
            sc = torch.cat([sc, sink.double()[:, None]], 1)
        w = torch.softmax(sc, -1)[:, :p + 1]
        want, size = torch.einsum("hj,jhd->hd", w, v), torch.einsum("hj,jhd->hd", w, v.abs())
        if gate is not None:
            s_g = torch.sigmoid(gate[t].double().view(nh, hdv))
            want, size = want * s_g, size * s_g
        # weights rounded to bf16 (half an ulp each) against values of that size, and the output's own rounding
        assert bool(((got[t] - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-5).all()), (t, p, s)


@pytest.mark.parametrize("spread", [1.0, 3.0])
def test_weights_round_no_worse_than_token_by_token(spread):
    """Few keys that hold most of a softmax, and many that share it: the error of the kernel for wide values is at most that
    of the general kernel, which keeps a token's largest weight at 1 (5% for other orders of summing)."""
    from cpmcu_amd import ops
    L, nh, hdk, hdv, page = 512, 16, 576, 512, 64
    g = torch.Generator().manual_seed(int(spread))
    k, q = torch.randn(L, 1, hdk, generator=g).to(torch.bfloat16), (spread * torch.randn(L, nh, hdk, generator=g)).to(torch.bfloat16)
    v = k[..., :hdv].contiguous()
    pools = []
    for x, keys in ((k, True), (v, False)):
        pool = torch.zeros(x.numel(), dtype=torch.bfloat16)
        pool[element_order(L, 1, x.shape[-1], keys).flatten()] = x.flatten()
        pools.append(pool.view(L // page, page, -1).to(DEV))
    pos, table = torch.arange(L, dtype=torch.int32, device=DEV), torch.arange(L // page, dtype=torch.int32, device=DEV)[None]
    slot, rows = torch.zeros_like(pos), q.view(L, -1).to(DEV)
    wide, general = (torch.empty(L, nh * hdv, device=DEV) for _ in range(2))
    shape = (nh, 1, hdk, hdv, hdk ** -0.5, *pools, table, page, pos, slot)
    ops.attention_wide_prefill(rows, wide, ops.prefill_tiles([L], 64 // nh, DEV), *shape, 0, 0, 0, None, 1, None, 0.0)
    ops.attention_general_mfma(rows, general, *shape)
    s = torch.einsum("thd,jd->htj", q.double(), k[:, 0].double()) * hdk ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    want = torch.matmul(torch.softmax(s, -1), v[:, 0].double()).transpose(0, 1).reshape(L, -1)
    off = [float((x.double().cpu() - want).norm()) for x in (wide, general)]
    assert off[0] <= 1.05 * off[1], off


@pytest.mark.parametrize("nh,nkv,spans,wide", [(32, 1, [(0, 160)], False), (32, 1, [(0, 161)], True), (32, 1, [(120, 160), (0, 1)], False),
                                               (32, 1, [(130, 170), (0, 1)], True), (8, 2, [(0, 64)] * 4, False), (8, 2, [(0, 65)] * 4, True),
                                               (32, 1, [(0, 100)] * 2 + [(0, 57)], True), (4, 4, [(0, 8)], True)])
def test_few_tokens_of_few_keys_take_the_general_kernel(nh, nkv, spans, wide, monkeypatch):
    """Both sides of the rule's borders (keys, workgroups, tokens, heads a kv head), each right."""
    from types import SimpleNamespace
    from cpmcu_amd import ops
    hdk, hdv, page = 128, 256, 64
    g = torch.Generator().manual_seed(sum(b for _, b in spans))
    width = max(-(-b // page) for _, b in spans)
    table = torch.arange(width * len(spans), dtype=torch.int32).view(len(spans), width)
    pools, kept = [], []
    for hd, keys in ((hdk, True), (hdv, False)):
        pool = torch.zeros(len(spans), width * page * nkv * hd, dtype=torch.bfloat16)
        rows = [torch.randn(b, nkv, hd, generator=g).to(torch.bfloat16) for _, b in spans]
        for s, x in enumerate(rows):
            pool[s, element_order(len(x), nkv, hd, keys).flatten()] = x.flatten()
        pools.append(pool.view(-1, page, nkv * hd).to(DEV))
        kept.append(rows)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(single_token=False, max_pos=max(b for _, b in spans) - 1, q_lens=[b - a for a, b in spans], extras={},
                          positions=i32([t for a, b in spans for t in range(a, b)]),
                          tok_slot=i32([s for s, (a, b) in enumerate(spans) for _ in range(a, b)]))
    n = sum(ctx.q_lens)
    q, out = torch.randn(n, nh, hdk, generator=g).to(torch.bfloat16), torch.full((n, nh * hdv), float("nan"), device=DEV)
    called = []
    for name in ("attention_wide_prefill", "attention_general_mfma"):
        monkeypatch.setattr(ops, name, lambda *a, _f=getattr(ops, name), _n=name, **k: (called.append(_n), _f(*a, **k)))
    ops.attention_any(q.view(n, -1).to(DEV), out, nh, nkv, hdk, hdv, hdk ** -0.5, *pools, table.to(DEV), page, ctx)
    assert called == ["attention_wide_prefill" if wide else "attention_general_mfma"]
    at = 0
    for s, (a, b) in enumerate(spans):
        k, v = (x[s].double().repeat_interleave(nh // nkv, 1) for x in kept)
        sc = torch.einsum("thd,jhd->htj", q[at:at + b - a].double(), k) * hdk ** -0.5
        sc.masked_fill_(torch.arange(b)[None] > torch.arange(a, b)[:, None], -math.inf)
        w = torch.softmax(sc, -1)
        want, size = (torch.einsum("htj,jhd->thd", w, x) for x in (v, v.abs()))
        got = out[at:at + b - a].double().cpu().view(b - a, nh, hdv)
        assert bool(((got - want).abs() <= 2.0 ** -8 * size + 1e-5).all()), s          # weights rounded to 8 bits
        at += b - a


@pytest.mark.parametrize("nh,nkv,hdk,hdv,opt", [(32, 1, 576, 512, {}), (8, 2, 128, 256, {"window": 40, "keep_first": 3, "gate": True}),
                                                (4, 4, 72, 132, {"sink": True, "softcap": 4.0}), (2, 1, 192, 512, {"chunk": 48, "out": torch.bfloat16})])
def test_infinities_reach_only_tokens_that_see_them(nh, nkv, hdk, hdv, opt):
    """Infinities and NaNs among the values of some tokens: tokens before them, or behind their window or chunk, have the
    results that they have without; the others what the sum over the keys that they see gives."""
    from cpmcu_amd import ops
    L, page, G = 203, 64, nh // nkv
    pool_hdk, pool_hdv, pages = -(-hdk // 64) * 64, -(-hdv // 16) * 16, 4
    g = torch.Generator().manual_seed(hdk)
    k, v = (torch.randn(L, nkv, hd, generator=g).to(torch.bfloat16) for hd in (hdk, hdv))
    for t, f, value in ((37, 5, math.inf), (38, 5, -math.inf), (90, hdv - 1, -math.inf), (91, 64, math.nan), (202, 0, math.inf)):
        v[t, t % nkv, f] = value
    q = torch.randn(L, nh, hdk, generator=g).to(torch.bfloat16)
    pools = []
    for x, hd, keys in ((k, pool_hdk, True), (v, pool_hdv, False)):
        flat = torch.full((pages * page * nkv * hd,), 0.0, dtype=torch.bfloat16)
        flat[element_order(L, nkv, hd, keys)[..., :x.shape[-1]].flatten()] = x.flatten()
        pools.append(flat.view(pages, page, -1).to(DEV))
    dev = lambda t: None if t is None else t.to(DEV)
    sink = torch.randn(nh, generator=g) if opt.get("sink") else None
    gate = torch.randn(L, nh * hdv, generator=g).to(torch.bfloat16) if opt.get("gate") else None
    chunk, window, keep, cap = (opt.get(t, 0) for t in ("chunk", "window", "keep_first", "softcap"))
    pos = torch.arange(L, dtype=torch.int32)
    out = torch.full((L, nh * hdv), 7.0, dtype=opt.get("out", torch.float32), device=DEV)
    ops.attention_wide_prefill(dev(q.view(L, -1)), out, ops.prefill_tiles([L], 64 // G, DEV), nh, nkv, hdk, hdv, hdk ** -0.5, *pools,
                               torch.arange(pages, dtype=torch.int32, device=DEV)[None], page, dev(pos), dev(torch.zeros_like(pos)),
                               chunk, window, keep, dev(sink), 1, dev(gate), float(cap))
    got = out.double().cpu().view(L, nh, hdv)
    kd, vd, j = k.double().repeat_interleave(G, 1), v.double().repeat_interleave(G, 1), torch.arange(L)
    for t in range(L):
        sees = (j <= t) & ((j // chunk == t // chunk) if chunk else ((t - j < window) | (j < keep)) if window else True)
        sc = torch.einsum("hd,jhd->hj", q[t].double(), kd[sees]) * hdk ** -0.5
        sc = cap * torch.tanh(sc / cap) if cap else sc
        if sink is not None:
            sc = torch.cat([sc, sink.double()[:, None]], 1)
        w = torch.softmax(sc, -1)[:, :int(sees.sum()), None]
        terms = w * vd[sees].transpose(0, 1)
        want, size = terms.sum(1), terms.abs().sum(1)
        if gate is not None:
            s_g = torch.sigmoid(gate[t].double().view(nh, hdv))
            want, size = want * s_g, size * s_g
        fine = torch.isfinite(want)
        assert torch.equal(got[t].isnan(), want.isnan()) and torch.equal(got[t][~fine].nan_to_num(0.0), want[~fine].nan_to_num(0.0)), t
        assert bool(((got[t] - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-5)[fine].all()), t


@pytest.fixture
def columns_128(monkeypatch):
    """Workgroups of 128 columns, tiles of twice the tokens."""
    from cpmcu_amd import ops
    wide, tiles = ops.attention_wide_prefill, ops.prefill_tiles
    monkeypatch.setattr(ops, "attention_wide_prefill", lambda *a, **k: wide(*a, **k, columns=128))
    monkeypatch.setattr(ops, "prefill_tiles", lambda lens, per, device: tiles(lens, 2 * per, device))


@pytest.mark.parametrize("nh,nkv,hdk,hdv,v_share,opt", [
    (32, 1, 576, 512, 1, {}), (32, 1, 576, 512, 1, {"window": 37, "sink": True, "gate": True}), (8, 2, 576, 260, 2, {"chunk": 48}),
    (64, 1, 520, 512, 1, {"softcap": 3.0, "out": torch.float32}), (6, 3, 568, 272, 3, {"window": 20, "keep_first": 5, "page": 32}),
    (2, 2, 576, 384, 1, {"page": 96, "sink": True})])
def test_wide_prompt_attention_of_128_columns(nh, nkv, hdk, hdv, v_share, opt, columns_128):
    """1 to 64 tokens a workgroup, tiles that end early, keys and values beside the cached sizes, every mask."""
    test_wide_prompt_attention(nh, nkv, hdk, 576, hdv, v_share, opt)


@pytest.mark.parametrize("spread", [1.0, 3.0])
def test_weights_of_128_columns_round_no_worse(spread, columns_128):
    test_weights_round_no_worse_than_token_by_token(spread)


@pytest.mark.parametrize("nh,nkv,hdk,hdv,opt", [(32, 1, 576, 512, {}), (8, 2, 520, 272, {"window": 40, "keep_first": 3, "gate": True}),
                                                (4, 4, 576, 260, {"sink": True, "softcap": 4.0}), (2, 1, 576, 512, {"chunk": 48, "out": torch.bfloat16})])
def test_infinities_in_128_columns(nh, nkv, hdk, hdv, opt, columns_128):
    test_infinities_reach_only_tokens_that_see_them(nh, nkv, hdk, hdv, opt)


def test_the_rule_of_128_columns():
    from cpmcu_amd import ops
    cus = ops.compute_units()
    most = -(-5 * cus // 4)                                                  # workgroups of 4 tokens of 32 heads
    assert ops.attention_wide_columns([4 * most], 32, 1, 576, 512) == 128 and ops.attention_wide_columns([4 * most - 4], 32, 1, 576, 512) == 64
    assert ops.attention_wide_columns([1] * most, 32, 1, 576, 512) == 128
    for other in ((32, 1, 512, 512), (32, 1, 576, 256), (6, 2, 576, 512)):
        assert ops.attention_wide_columns([4 * most * 4], *other) == 64
    with pytest.raises(ops.KernelError, match="128 columns|columns a workgroup"):
        x = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16, device=DEV)
        i = lambda *shape: torch.zeros(*shape, dtype=torch.int32, device=DEV)
        ops.attention_wide_prefill(x(1, 128), x(1, 256), torch.tensor([[0, 1]], dtype=torch.int32, device=DEV), 1, 1, 128, 256, 1.0, x(1, 64, 128), x(1, 64, 256),
                                   i(1, 1), 64, i(1), i(1), columns=128)


@pytest.mark.parametrize("spans,mask,columns", [
    ([(0, 161 + s) for s in range(8)], {}, 128), ([(0, 163)] * 7, {}, 64),                       # 331 and 287 workgroups of 4 tokens
    ([(0, 161 + s) for s in range(8)] + [(900, 905)], {}, 64), ([(400, 563)] * 8, {"window": 130, "keep_first": 3}, 128)])
def test_columns_and_tiles_of_a_step_go_together(spans, mask, columns, monkeypatch):
    """A step over a latent on both sides of the rule of 128 columns: the tiles are cut for the columns that the kernel is
    launched with, so that every token's output is written."""
    from types import SimpleNamespace
    from cpmcu_amd import ops
    nh, hdk, hdv, page = 32, 576, 512, 64
    monkeypatch.setattr(ops, "_cu_count", 256)
    g = torch.Generator().manual_seed(len(spans))
    width = max(-(-b // page) for _, b in spans)
    pools, kept = [torch.zeros(len(spans), width * page * hd, dtype=torch.bfloat16) for hd in (hdk, hdv)], []
    for s, (_, b) in enumerate(spans):
        kept.append([torch.randn(b, 1, hd, generator=g).to(torch.bfloat16) for hd in (hdk, hdv)])
        for pool, x, keys in zip(pools, kept[-1], (True, False)):
            pool[s, element_order(b, 1, x.shape[-1], keys).flatten()] = x.flatten()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(single_token=False, max_pos=max(b for _, b in spans) - 1, q_lens=[b - a for a, b in spans],
                          kv_lens=[b for _, b in spans], extras={}, positions=i32([t for a, b in spans for t in range(a, b)]),
                          tok_slot=i32([s for s, (a, b) in enumerate(spans) for _ in range(a, b)]))
    n, launched, wide = sum(ctx.q_lens), [], ops.attention_wide_prefill
    monkeypatch.setattr(ops, "attention_wide_prefill", lambda *a: (launched.append((int(a[2][:, 1].max()), a[-1])), wide(*a)))
    q, out = torch.randn(n, nh, hdk, generator=g).to(torch.bfloat16), torch.full((n, nh * hdv), float("nan"), device=DEV)
    ops.attention_any(q.view(n, -1).to(DEV), out, nh, 1, hdk, hdv, hdk ** -0.5, *(p.view(-1, page, p.shape[1] // (width * page)).to(DEV) for p in pools),
                      torch.arange(width * len(spans), dtype=torch.int32, device=DEV).view(len(spans), width), page, ctx, **mask)
    assert launched == [(columns // nh, columns)]
    at = 0
    for s, (a, b) in enumerate(spans):
        k, v = (x[:, 0].double().to(DEV) for x in kept[s])
        sc = (q[at:at + b - a].double().to(DEV).view(-1, hdk) @ k.T).view(b - a, nh, b) * hdk ** -0.5
        p, j = torch.arange(a, b, device=DEV)[:, None], torch.arange(b, device=DEV)[None]
        hidden = (j > p) | ((p - j >= mask["window"]) & (j >= mask["keep_first"]) if mask else False)
        w = torch.softmax(sc.masked_fill(hidden[:, None], -math.inf), -1)
        want, size = ((w.view(-1, b) @ x).view(b - a, nh * hdv) for x in (v, v.abs()))
        # weights rounded to bf16 (half an ulp each) against values of that size
        assert bool(((out[at:at + b - a].double() - want).abs() <= 2.0 ** -8 * size + 1e-5).all()), s
        at += b - a


def test_outputs_off_16_byte_borders_take_the_general_kernel():
    from types import SimpleNamespace
    from cpmcu_amd import ops
    L, hdk, hdv, page = 200, 64, 132, 64
    g = torch.Generator().manual_seed(5)
    k, v, q = (torch.randn(L, 1, hd, generator=g).to(torch.bfloat16) for hd in (hdk, hdv, hdk))
    pools = []
    for x, hd, keys in ((k, hdk, True), (v, 144, False)):
        flat = torch.zeros(4 * page * hd, dtype=torch.bfloat16)
        flat[element_order(L, 1, hd, keys)[..., :x.shape[-1]].flatten()] = x.flatten()
        pools.append(flat.view(4, page, -1).to(DEV))
    pos = torch.arange(L, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(single_token=False, max_pos=L - 1, q_lens=[L], extras={}, positions=pos, tok_slot=torch.zeros_like(pos))
    out = torch.zeros(L + 1, hdv, dtype=torch.bfloat16, device=DEV)[1:]                 # 264 bytes on
    ops.attention_any(q.view(L, -1).to(DEV), out, 1, 1, hdk, hdv, 0.1, *pools, torch.arange(4, dtype=torch.int32, device=DEV)[None],
                      page, ctx)
    s = 0.1 * q[:, 0].double() @ k[:, 0].double().T
    w = torch.softmax(s.masked_fill(torch.ones(L, L, dtype=torch.bool).triu(1), -math.inf), -1)
    want, size = w @ v[:, 0].double(), w @ v[:, 0].double().abs()
    # weights rounded to bf16 against values of that size, and the output's own rounding
    assert bool(((out.double().cpu() - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-5).all())
