"""Experts grouped into tiles: row counts at the edges of tiles, of 16 rows and of the rule for wide tiles; widths that end
inside a piece of 64 columns or a tile of features (GPU)."""
import launched
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows: how many pairs each expert gets (the last one none); `top` 1 makes that exact
@pytest.mark.parametrize("rows", [[1], [16, 17], [32, 33, 1], [64, 65], [128, 129, 96, 97], [257, 5], [1030, 3, 0, 500]])
@pytest.mark.parametrize("H,F", [(8, 8), (72, 136), (200, 56)])
@pytest.mark.parametrize("gated", [True, False])
def test_tiles_of_every_fill(rows, H, F, gated):
    from cpmcu_amd import ops
    E, n = len(rows) + 1, sum(rows)
    g = torch.Generator(device=DEV).manual_seed(n + H + F)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(rows)])
    idx = idx[torch.randperm(n, generator=torch.Generator().manual_seed(n))].to(DEV)[:, None].contiguous()
    h = torch.randn(n, H, generator=g, device=DEV).to(torch.bfloat16)
    up = torch.randn(E, F * (2 if gated else 1), H, generator=g, device=DEV).to(torch.bfloat16)
    down = torch.randn(E, H, F, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.rand(n, 1, generator=g, device=DEV)
    tiles = ops.moe_tiles(n, 1, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    act = torch.full((n, 1, F), float("nan"), dtype=torch.bfloat16, device=DEV)
    y = torch.full((n, 1, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((n, H), float("nan"), device=DEV)
    ops.moe_experts_mfma(h, up, down, idx, w, out, act, y, i32(tiles * ops.MOE_TILE), i32(tiles), i32(1), gated=gated,
                         activation="silu" if gated else "relu_squared")
    e = idx[:, 0].long()
    half, sums = 2.0 ** -8, 2.0 ** -23
    z = torch.einsum("nk,nfk->nf", h.double(), up.double()[e])
    mag = torch.einsum("nk,nfk->nf", h.double().abs(), up.double().abs()[e])
    off = H * sums * mag                                             # float sums in any order
    if gated:
        a, u = z[:, :F], z[:, F:]
        want = torch.nn.functional.silu(a) * u
        off = 1.1 * off[:, :F] * u.abs() + (a.abs() + off[:, :F]) * off[:, F:]      # |silu'| <= 1.1
    else:
        want = torch.relu(z) ** 2
        off = 2 * z.abs() * off + off ** 2
    assert bool(((act[:, 0].double() - want).abs() <= off + (half + 8 * sums) * want.abs() + 1e-30).all())
    got = act[:, 0].double()                                         # the second product of what the first one wrote
    ref = torch.einsum("nf,nhf->nh", got, down.double()[e])
    off = F * sums * torch.einsum("nf,nhf->nh", got.abs(), down.double().abs()[e])
    off = off + half * (ref.abs() + off)
    assert bool(((out.double() - w.double() * ref).abs() <= w.double() * off + 2 * sums * ref.abs() + 1e-30).all())


@pytest.mark.parametrize("H,F", [(8, 64), (64, 104), (72, 200), (128, 128), (200, 264), (264, 72), (192, 320)])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("offset", [0, 1])
def test_tiles_of_128_rows(H, F, gated, offset):
    """Steps of 48 pairs an expert or more: fills at the edges of every form (the last expert none), one, two, three and more
    pieces of 64 columns, whole and ragged, features that end inside a tile; pair outputs off 16-byte borders, and a row that
    is no number, which reaches no other."""
    from cpmcu_amd import ops
    rows = [1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 256, 257, 300, 513]
    E, n = len(rows) + 1, sum(rows)
    assert n >= 48 * E
    g = torch.Generator(device=DEV).manual_seed(H + F)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(rows)])
    idx = idx[torch.randperm(n, generator=torch.Generator().manual_seed(n))].to(DEV)[:, None].contiguous()
    h = torch.randn(n, H, generator=g, device=DEV).to(torch.bfloat16)
    h[7] = float("nan")
    up = torch.randn(E, F * (2 if gated else 1), H, generator=g, device=DEV).to(torch.bfloat16)
    down = torch.randn(E, H, F, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.rand(n, 1, generator=g, device=DEV)
    tiles = ops.moe_tiles(n, 1, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    act = torch.full((n, 1, F), 7.0, dtype=torch.bfloat16, device=DEV)
    y = torch.full((n * H + offset + 1,), 7.0, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(n, H, device=DEV)
    ops.moe_experts_mfma(h, up, down, idx, w, out, act, y[offset:offset + n * H].view(n, 1, H), i32(tiles * ops.MOE_TILE), i32(tiles),
                         i32(1), gated=gated, activation="silu" if gated else "relu_squared")
    assert bool((y[:offset] == 7).all()) and bool((y[offset + n * H:] == 7).all())
    assert not gated or (bool(act[7].isnan().all()) and bool(out[7].isnan().all()))      # (max(z, 0) of no number is 0)
    half, sums = 2.0 ** -8, 2.0 ** -23
    for e in range(E):
        mine = (idx[:, 0] == e).nonzero()[:, 0]
        mine = mine[mine != 7]
        x, u = h[mine].double(), up[e].double()
        z, off = x @ u.T, H * sums * (x.abs() @ u.abs().T)           # float sums in any order
        if gated:
            a, b = z[:, :F], z[:, F:]
            want = torch.nn.functional.silu(a) * b
            off = 1.1 * off[:, :F] * b.abs() + (a.abs() + off[:, :F]) * off[:, F:]      # |silu'| <= 1.1
        else:
            want, off = torch.relu(z) ** 2, 2 * z.abs() * off + off ** 2
        got = act[mine, 0].double()
        assert bool(((got - want).abs() <= off + (half + 8 * sums) * want.abs() + 1e-30).all()), (e, rows[e] if e < len(rows) else 0)
        ref, off = got @ down[e].double().T, F * sums * (got.abs() @ down[e].double().abs().T)
        off = off + half * (ref.abs() + off)
        v = w[mine].double()
        assert bool(((out[mine].double() - v * ref).abs() <= v * off + 2 * sums * ref.abs() + 1e-30).all()), e


@pytest.mark.parametrize("H,F", [(72, 136), (200, 56), (1024, 136), (1096, 264)])
def test_experts_without_a_gate_of_few_tokens(H, F):
    """Up to 64 tokens, whose first product of 1,024 columns and more runs on tiles of 64 rows of another kernel; an expert that is every choice of every
    token has more rows than there are tokens."""
    from cpmcu_amd import ops
    E, n, top = 9, 40, 3
    g = torch.Generator(device=DEV).manual_seed(H)
    idx = torch.randint(0, E, (n, top), generator=torch.Generator().manual_seed(1), dtype=torch.int32)
    idx[:31] = 4
    idx = idx.to(DEV)
    h = torch.randn(n, H, generator=g, device=DEV).to(torch.bfloat16)
    up = torch.randn(E, F, H, generator=g, device=DEV).to(torch.bfloat16)
    down = torch.randn(E, H, F, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.rand(n, top, generator=g, device=DEV)
    tiles = ops.moe_tiles(n, top, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    act, y = (torch.full((n, top, k), float("nan"), dtype=torch.bfloat16, device=DEV) for k in (F, H))
    ops.moe_experts_mfma(h, up, down, idx, w, torch.empty(n, H, device=DEV), act, y, i32(tiles * ops.MOE_TILE), i32(tiles), i32(1),
                         gated=False, activation="relu_squared")
    e = idx.long()
    z = torch.einsum("nh,nkfh->nkf", h.double(), up.double()[e])
    off = H * 2.0 ** -23 * torch.einsum("nh,nkfh->nkf", h.double().abs(), up.double().abs()[e])
    want, off = torch.relu(z) ** 2, 2 * z.abs() * off + off ** 2
    assert bool(((act.double() - want).abs() <= off + (2.0 ** -8 + 2.0 ** -20) * want.abs() + 1e-30).all())
    ref = torch.einsum("nkf,nkhf->nkh", act.double(), down.double()[e])
    off = F * 2.0 ** -23 * torch.einsum("nkf,nkhf->nkh", act.double().abs(), down.double().abs()[e])
    assert bool(((y.double() - ref).abs() <= off + 2.0 ** -8 * (ref.abs() + off) + 1e-30).all())


def forms(E, pairs, H, F, gated, top=1):
    """(first product's, second's) kernel of a step of so many pairs, one more of the first expert than of others at most."""
    from cpmcu_amd import ops
    n = pairs // top
    assert n * top == pairs
    idx = (torch.arange(pairs, dtype=torch.int32, device=DEV) % E).view(n, top)
    rnd = lambda *shape: torch.randn(*shape, device=DEV).to(torch.bfloat16)
    h, up, down, w = rnd(n, H), rnd(E, F * (2 if gated else 1), H), rnd(E, H, F), torch.rand(n, top, device=DEV)
    tiles = ops.moe_tiles(n, top, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    scratch = rnd(n, top, F), rnd(n, top, H), i32(tiles * ops.MOE_TILE), i32(tiles), i32(1)
    names = launched.kernels(lambda: ops.moe_experts_mfma(h, up, down, idx, w, torch.empty(n, H, device=DEV), *scratch, gated=gated,
                                                          activation="silu" if gated else "relu_squared"))
    return tuple("wide" if "moe_wide" in name else "tile" for name in names if "moe_wide" in name or "moe_tile" in name)


@pytest.mark.parametrize("E,pairs,F,gated,want", [
    (8, 384, 72, True, "wide"), (8, 383, 72, True, "tile"), (8, 383, 72, False, "tile"),
    (64, 1536, 1024, True, "wide"), (64, 1535, 1024, True, "tile"), (64, 1536, 960, True, "tile"), (64, 1536, 2048, False, "wide"),
    (64, 1536, 1920, False, "tile"), (32, 1408, 512, True, "tile"), (8, 352, 512, False, "tile")])
def test_the_rule_of_wide_tiles(E, pairs, F, gated, want):
    """48 pairs an expert, or 24 where the first product has 1,024 workgroups."""
    assert forms(E, pairs, 64, F, gated) == (want, want)


@pytest.mark.parametrize("E,n,top,H,F,want", [
    (8, 64, 2, 1024, 512, "wide"), (8, 64, 2, 1016, 512, "tile"), (8, 65, 2, 1024, 512, "tile"), (16, 64, 1, 1024, 2048, "wide"),
    (16, 64, 1, 1024, 2056, "tile"), (64, 24, 6, 1024, 2112, "tile"), (64, 4, 6, 1024, 1280, "wide"), (64, 4, 6, 1024, 1408, "tile")])
def test_the_rule_of_first_products_without_a_gate(E, n, top, H, F, want):
    """Up to 64 tokens of 1,024 columns or more, a workgroup a CU at most."""
    assert forms(E, n * top, H, F, False, top) == (want, "tile")


@pytest.mark.parametrize("H,F", [(72, 136), (264, 72)])
@pytest.mark.parametrize("gated", [True, False])
def test_full_and_split_tiles_of_64_rows(H, F, gated):
    """Experts of 64 to 300 rows among others without any: below the rule of wide tiles, a tile of 64 rows full, two and
    three of them."""
    from cpmcu_amd import ops
    rows = [64, 65, 63, 129, 128, 300] + [0] * 12
    E, n = len(rows), sum(rows)
    assert n < 48 * E
    g = torch.Generator(device=DEV).manual_seed(H)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(rows)])
    idx = idx[torch.randperm(n, generator=torch.Generator().manual_seed(n))].to(DEV)[:, None].contiguous()
    h, up, down = (torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16) for s in ((n, H), (E, F * (2 if gated else 1), H), (E, H, F)))
    w = torch.rand(n, 1, generator=g, device=DEV)
    tiles = ops.moe_tiles(n, 1, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    act, y = (torch.full((n, 1, k), float("nan"), dtype=torch.bfloat16, device=DEV) for k in (F, H))
    ops.moe_experts_mfma(h, up, down, idx, w, torch.empty(n, H, device=DEV), act, y, i32(tiles * ops.MOE_TILE), i32(tiles), i32(1),
                         gated=gated, activation="silu" if gated else "relu_squared")
    half, sums = 2.0 ** -8, 2.0 ** -23
    for e in range(6):
        mine = (idx[:, 0] == e).nonzero()[:, 0]
        x, u, got = h[mine].double(), up[e].double(), act[mine, 0].double()
        z, off = x @ u.T, H * sums * (x.abs() @ u.abs().T)           # float sums in any order
        if gated:
            a, b = z[:, :F], z[:, F:]
            want = torch.nn.functional.silu(a) * b
            off = 1.1 * off[:, :F] * b.abs() + (a.abs() + off[:, :F]) * off[:, F:]      # |silu'| <= 1.1
        else:
            want, off = torch.relu(z) ** 2, 2 * z.abs() * off + off ** 2
        assert bool(((got - want).abs() <= off + (half + 8 * sums) * want.abs() + 1e-30).all()), rows[e]
        ref, off = got @ down[e].double().T, F * sums * (got.abs() @ down[e].double().abs().T)
        assert bool(((y[mine, 0].double() - ref).abs() <= off + half * (ref.abs() + off) + 1e-30).all()), rows[e]


@pytest.mark.parametrize("rows", [[80, 112], [81, 79, 97], [65, 113, 64]])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("H,F", [(136, 72), (264, 200)])
def test_pair_outputs_at_any_address(rows, gated, H, F):
    """Rows between the forms of wide tiles; pair outputs off 16-byte borders, which are stored element by element: the same."""
    from cpmcu_amd import ops
    E, n = len(rows), sum(rows)
    g = torch.Generator(device=DEV).manual_seed(n + H)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(rows)]).to(DEV)[:, None].contiguous()
    h = torch.randn(n, H, generator=g, device=DEV).to(torch.bfloat16)
    up = torch.randn(E, F * (2 if gated else 1), H, generator=g, device=DEV).to(torch.bfloat16)
    down = torch.randn(E, H, F, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.rand(n, 1, generator=g, device=DEV)
    tiles = ops.moe_tiles(n, 1, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)

    def run(offset):
        act = torch.full((n, 1, F), float("nan"), dtype=torch.bfloat16, device=DEV)
        y = torch.full((n * H + offset + 1,), float("nan"), dtype=torch.bfloat16, device=DEV)
        out = torch.empty(n, H, device=DEV)
        ops.moe_experts_mfma(h, up, down, idx, w, out, act, y[offset:offset + n * H].view(n, 1, H), i32(tiles * ops.MOE_TILE),
                             i32(tiles), i32(1), gated=gated, activation="silu" if gated else "relu_squared")
        assert bool(y[:offset].isnan().all()) and bool(y[offset + n * H:].isnan().all())
        return out, act

    (out, act), (out1, act1) = run(0), run(1)
    assert bool(out.isfinite().all()) and torch.equal(out, out1) and torch.equal(act, act1)
    e = idx[:, 0].long()
    want = torch.einsum("nf,nhf->nh", act[:, 0].double(), down.double()[e])
    mag = torch.einsum("nf,nhf->nh", act[:, 0].double().abs(), down.double().abs()[e])
    off = F * 2.0 ** -23 * mag                                       # float sums in any order, one rounding to bf16
    off = off + 2.0 ** -8 * (want.abs() + off)
    assert bool(((out.double() - w.double() * want).abs() <= w.double() * off + 2.0 ** -22 * want.abs() + 1e-30).all())


@pytest.mark.parametrize("top", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("H", [8, 2048, 2056])
@pytest.mark.parametrize("shared_dtype", [None, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("joined", [False, True])
def test_sum_of_a_tokens_experts(top, H, shared_dtype, joined):
    """The sum over a token's experts (identity experts among them), the shared expert and the layer's other result, for every
    number that has its own form; pair outputs off 16-byte borders take the general one: the same."""
    from cpmcu_amd import ops
    E, F, n = 5, 16, 33
    g = torch.Generator(device=DEV).manual_seed(top + H)
    rnd = lambda *shape, dtype=torch.bfloat16: torch.randn(*shape, generator=g, device=DEV).to(dtype)
    h, up, down = rnd(n, H), rnd(E, 2 * F, H) * 0.1, rnd(E, H, F)
    idx = torch.randint(0, E + 2, (n, top), generator=torch.Generator().manual_seed(top), dtype=torch.int32).to(DEV)
    w = torch.rand(n, top, generator=g, device=DEV)
    shared = None if shared_dtype is None else rnd(2, n, H, dtype=shared_dtype) if shared_dtype == torch.float32 else rnd(n, H)
    sg = None if shared is None else torch.rand(n, generator=g, device=DEV)
    x0, a, bias = rnd(n, H, dtype=torch.float32), rnd(3, n, H, dtype=torch.float32), rnd(H, dtype=torch.float32)
    tiles = ops.moe_tiles(n, top, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)

    def run(offset):
        act = torch.empty(n, top, F, dtype=torch.bfloat16, device=DEV)
        y = torch.full((n * top * H + offset,), float("nan"), dtype=torch.bfloat16, device=DEV)[offset:].view(n, top, H)
        x, copy, out = x0.clone(), torch.empty(n, H, dtype=torch.bfloat16, device=DEV), torch.empty(n, H, device=DEV)
        join = ops.Join(x, a, bias, copy) if joined else None
        ops.moe_experts_mfma(h, up, down, idx, w, None if joined else out, act, y, i32(tiles * ops.MOE_TILE), i32(tiles), i32(1), shared, sg, join=join)
        return (x if joined else out), copy, y

    got, copy, y = run(0)
    other, copy1, _ = run(1)
    assert torch.equal(got, other)
    rows = torch.where((idx < E)[..., None], y.double(), h.double()[:, None])
    terms = [w.double()[..., None] * rows]
    if shared is not None:
        terms.append((sg.double()[:, None] * (shared.double().sum(0) if shared.dim() == 3 else shared.double()))[:, None])
    if joined:
        terms += [x0.double()[:, None], a.double().transpose(0, 1), bias.double().expand(n, H)[:, None]]
        assert torch.equal(copy, got.to(torch.bfloat16)) and torch.equal(copy, copy1)
    terms = torch.cat(terms, 1)
    mag = terms.abs().sum(1) + (0 if shared is None or shared.dim() < 3 else sg.double()[:, None] * shared.double().abs().sum(0))
    assert bool(((got.double() - terms.sum(1)).abs() <= (terms.shape[1] + 3) * 2.0 ** -23 * mag).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gated_experts_of_more_pairs_than_a_grid_dimension(dtype):
    """33,003 pairs: the launch has two layers of 32,768; identity experts write nothing."""
    from cpmcu_amd import ops
    n, top, E, H, F = 11001, 3, 7, 16, 24
    g = torch.Generator(device=DEV).manual_seed(3)
    h, gu = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((n, H), (E, 2 * F, H)))
    idx = torch.randint(0, E + 2, (n, top), generator=torch.Generator().manual_seed(4), dtype=torch.int32).to(DEV)
    act = torch.full((n, top, F), float("nan"), dtype=dtype, device=DEV)
    ops.moe_gated(h, gu, idx, act)
    real = idx < E
    assert torch.equal(act.isnan(), ~real[..., None].expand_as(act))
    y = torch.matmul(gu.double(), h.double().T).permute(2, 0, 1)                          # [n, E, 2F]
    y = torch.gather(y, 1, idx.long().clamp(max=E - 1)[..., None].expand(n, top, 2 * F))
    want = torch.nn.functional.silu(y[..., :F]) * y[..., F:]
    # H float sums of both factors, and the output's own rounding
    mag = torch.gather(torch.matmul(gu.double().abs(), h.double().abs().T).permute(2, 0, 1), 1, idx.long().clamp(max=E - 1)[..., None].expand(n, top, 2 * F))
    off = (H + 6) * 2.0 ** -24 * (1.1 * mag[..., :F] * y[..., F:].abs() + mag[..., F:] * y[..., :F].abs() + want.abs()) + 1e-30
    off = off + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * want.abs()
    assert bool(((act.double() - want).abs() <= off)[real].all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 3, 16, 37])
@pytest.mark.parametrize("H", [8, 120, 128, 136, 264, 1000])
def test_down_products_of_any_number_of_column_blocks(n, H, dtype):
    """Blocks of 16 columns are dealt to the XCDs by eights, what is left over in order: 1, 8, 9, 17 and 63 blocks, all written."""
    from cpmcu_amd import ops
    E, F, top = 5, 40, 3
    g = torch.Generator(device=DEV).manual_seed(n + H)
    act, down = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((n, top, F), (E, H, F)))
    idx = torch.randint(0, E, (n, top), generator=torch.Generator().manual_seed(n), dtype=torch.int32).to(DEV)
    w = torch.rand(n, top, generator=g, device=DEV)
    out = torch.full((n, H), float("nan"), device=DEV)
    ops.moe_down(act, down, idx, w, out)
    terms = w.double()[..., None] * torch.matmul(down.double()[idx.long()], act.double()[..., None])[..., 0]
    mag = w.double()[..., None] * torch.matmul(down.double().abs()[idx.long()], act.double().abs()[..., None])[..., 0]
    assert bool(((out.double() - terms.sum(1)).abs() <= (F + top + 2) * 2.0 ** -24 * mag.sum(1)).all())
