"""Routed experts of many rows on the tiles of large products: fills at the edges of every form, features that end inside a tile, rows
beyond one tile, and what the rule gives to the other kernels (GPU)."""
import launched
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# 16 experts at least; fills at the edges of 32 rows and of tiles of 224, one expert without rows
ROWS = [1, 31, 33, 95, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 257, 448, 449, 700, 1345, 0]


def operands(rows, H, F, gated, seed, top=1):
    E, pairs = len(rows), sum(rows)
    g = torch.Generator(device=DEV).manual_seed(seed)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(rows)])
    idx = idx[torch.randperm(pairs, generator=torch.Generator().manual_seed(seed))].to(DEV).view(-1, top).contiguous()
    n = pairs // top
    h = torch.randn(n, H + 16, generator=g, device=DEV).to(torch.bfloat16)[:, 8:H + 8]          # rows apart, 16 bytes in
    up = torch.randn(E, F * (2 if gated else 1), H, generator=g, device=DEV).to(torch.bfloat16)
    down = torch.randn(E, H, F, generator=g, device=DEV).to(torch.bfloat16)
    return E, n, h, up, down, idx, torch.rand(n, top, generator=g, device=DEV)


def call(E, n, h, up, down, idx, w, act, y, out, gated, activation):
    from cpmcu_amd import ops
    tiles = ops.moe_tiles(n, idx.shape[1], E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    ops.moe_experts_mfma(h, up, down, idx, w, out, act, y, i32(tiles * ops.MOE_TILE), i32(tiles), i32(1), gated=gated, activation=activation)


@pytest.mark.parametrize("H,F,activation", [(4096, 1088, "silu"), (2048, 1600, "relu_squared"), (1600, 2048, ("clamped_swish", 7.0)),
                                            (4160, 832, "gelu_tanh"), (4096, 1088, "plain_silu")])
def test_every_fill(H, F, activation):
    gated = activation not in ("relu_squared", "plain_silu")
    top = 2
    rows = list(ROWS)
    rows[0] += sum(rows) % top
    E, n, h, up, down, idx, w = operands(rows, H, F, gated, H + F, top)
    assert n * top >= 64 * E and n * top * H * F >= 14e9
    h = h * 2 ** -3
    h[7] = float("nan")
    act = torch.full((n * top + 1, F), 7.0, dtype=torch.bfloat16, device=DEV)
    y = torch.full((n * top + 1, H), 7.0, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(n, H, device=DEV)
    run = lambda: call(E, n, h, up, down, idx, w, act[:-1].view(n, top, F), y[:-1].view(n, top, H), out, gated,
                       "silu" if activation == "plain_silu" else activation)
    names = launched.kernels(run)
    assert sum("moe_product" in name for name in names) == 2 and not any("moe_wide" in name or "moe_tile" in name for name in names)
    assert bool((act[-1] == 7).all()) and bool((y[-1] == 7).all())
    if activation in ("silu", "gelu_tanh", "plain_silu"):               # (the others' min and max of no number are numbers)
        assert bool(act[14:16].isnan().all()) and bool(out[7].isnan().all())
    first = act.clone(), y.clone()
    for _ in range(3):                                                  # another order of rows and tasks: the same numbers
        run()
        assert torch.equal(act.view(torch.int16), first[0].view(torch.int16)) and torch.equal(y.view(torch.int16), first[1].view(torch.int16))
    half, sums = 2.0 ** -8, 2.0 ** -23
    flat = idx.flatten()
    for e in range(E):
        mine = (flat == e).nonzero()[:, 0]
        mine = mine[mine // top != 7]
        x, u = h[mine // top].double(), up[e].double()
        z, off = x @ u.T, H * sums * (x.abs() @ u.abs().T)              # float sums in any order
        a = z[:, :F]
        # (the exponential's argument is rounded to 2^-24 of itself: |a| e^-|a| < 0.4 of a gate's value; |act'| <= 1.13)
        fast = 16 * sums * (1 + a.abs())
        if gated:
            b, ob = z[:, F:], off[:, F:]
            if activation == "silu":
                v, slope = torch.nn.functional.silu(a), 1.1
            elif activation == "gelu_tanh":
                v, slope, fast = torch.nn.functional.gelu(a, approximate="tanh"), 1.13, 16 * sums * (1 + 2 * a.abs() + 0.1 * a.abs() ** 3)
            else:
                a, b = a.clamp(max=7.0), b.clamp(-7.0, 7.0) + 1
                v, slope = a * torch.sigmoid(1.702 * a), 1.1
            want = v * b
            off = slope * off[:, :F] * b.abs() + (a.abs() + off[:, :F]) * ob + fast * want.abs()
        elif activation == "plain_silu":
            want = torch.nn.functional.silu(a)
            off = 1.1 * off + fast * want.abs()
        else:
            want, off = torch.relu(z) ** 2, 2 * z.abs() * off + off ** 2
        got = act[mine].double()
        assert bool(((got - want).abs() <= off + (half + 8 * sums) * want.abs() + 1e-30).all()), (e, rows[e])
        ref, off = got @ down[e].double().T, F * sums * (got.abs() @ down[e].double().abs().T)
        assert bool(((y[mine].double() - ref).abs() <= off + half * (ref.abs() + off) + 1e-30).all()), (e, rows[e])


@pytest.mark.parametrize("E,pairs,H,F,want", [
    (16, 4096, 2048, 1728, "product"), (16, 4096, 2048, 1664, "wide"), (15, 4500, 2048, 1728, "wide"), (72, 64 * 72, 2048, 1536, "product"),
    (72, 64 * 72 - 1, 2048, 1536, "wide"), (16, 4096, 2048, 1736, "wide"), (16, 8192, 4096, 448, "wide"), (16, 8192, 4096, 512, "product"),
    (64, 7872, 1536, 1792, "product"), (64, 7552, 1536, 1792, "wide")])
@pytest.mark.parametrize("gated", [True, False])
def test_the_rule(E, pairs, H, F, want, gated):
    """64 pairs an expert, 16 experts, 14e9 products (21e9 of fewer than 1,600 columns); whole pieces of 64 columns, 8 of them."""
    rows = [pairs // E + (e < pairs % E) for e in range(E)]
    E, n, h, up, down, idx, w = operands(rows, H, F, gated, F)
    act, y = (torch.empty(n, 1, k, dtype=torch.bfloat16, device=DEV) for k in (F, H))
    names = launched.kernels(lambda: call(E, n, h, up, down, idx, w, act, y, torch.empty(n, H, device=DEV), gated, "silu" if gated else "relu_squared"))
    assert ["product" if "moe_product" in x else "wide" for x in names if "moe_product" in x or "moe_wide" in x or "moe_tile" in x] == [want] * 2


def test_pair_outputs_off_16_byte_borders():
    """Pair outputs may start anywhere: such a call keeps the other kernel, with the same numbers."""
    rows = [260] * 16
    E, n, h, up, down, idx, w = operands(rows, 2048, 1728, True, 5)
    act = torch.empty(n, 1, 1728, dtype=torch.bfloat16, device=DEV)
    y = torch.full((n * 2048 + 2,), 7.0, dtype=torch.bfloat16, device=DEV)
    out = [torch.empty(n, 2048, device=DEV) for _ in range(2)]
    for i, o in enumerate(out):
        names = launched.kernels(lambda: call(E, n, h, up, down, idx, w, act, y[i:i + n * 2048].view(n, 1, 2048), o, True, "silu"))
        assert sum("moe_product" in x for x in names) == (0 if i else 2)
    assert float((out[0] - out[1]).norm()) <= 2.0 ** -8 * float(out[0].norm())


def test_inside_a_captured_graph():
    """Replays start from counters that the graph itself clears."""
    rows = [200 + 20 * e for e in range(16)]
    E, n, h, up, down, idx, w = operands(rows, 2048, 1728, True, 9)
    from cpmcu_amd import ops
    tiles = ops.moe_tiles(n, 1, E)
    i32 = lambda k: torch.empty(k, dtype=torch.int32, device=DEV)
    scratch = [torch.empty(n, 1, k, dtype=torch.bfloat16, device=DEV) for k in (1728, 2048)] + [i32(tiles * ops.MOE_TILE), i32(tiles), i32(1)]
    out = torch.empty(n, 2048, device=DEV)
    run = lambda: ops.moe_experts_mfma(h, up, down, idx, w, out, *scratch)
    run()
    torch.cuda.synchronize()
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        run()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", ("clamped_swish", 7.0), "plain_silu", "plain_gelu_tanh", "relu_squared"])
def test_the_bits_of_the_other_kernel(activation):
    """The same sums in the same order, the same nonlinearity in float: what the tiles of 128 rows give, to the last bit."""
    gated = not str(activation).startswith(("plain", "relu"))
    E, n, h, up, down, idx, w = operands([260, 300, 129, 700] * 4, 2048, 1728, gated, 11)
    h = h * 2.0 ** -4
    act = [torch.empty(n, 1, 1728, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    y = torch.full((2, n * 2048 + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    out = [torch.empty(n, 2048, device=DEV) for _ in range(2)]
    for i in range(2):                                                  # off its 16-byte border y keeps the other kernel
        run = lambda: call(E, n, h, up, down, idx, w, act[i], y[i, i:i + n * 2048].view(n, 1, 2048), out[i], gated, str(activation).removeprefix("plain_")
                           if isinstance(activation, str) else activation)
        assert sum("moe_product" in x for x in launched.kernels(run)) == (0 if i else 2)
    assert torch.equal(act[0], act[1]) and torch.equal(y[0, :n * 2048], y[1, 1:n * 2048 + 1]) and torch.equal(out[0], out[1])


def test_identity_experts():
    """Pairs of identity experts have no tiles; the rest of an uneven load, and an expert without rows, keep their places."""
    E, H, F, top, n = 20, 2048, 1728, 4, 1500
    g = torch.Generator(device=DEV).manual_seed(2)
    load = torch.cat([torch.arange(1, E + 9, device=DEV, dtype=torch.float32) ** 2])        # the last 8 columns: identity experts
    load[7] = 0
    idx = torch.multinomial(load.expand(n, -1), top, generator=g).to(torch.int32)
    h = torch.randn(n, H, generator=g, device=DEV).to(torch.bfloat16)
    up = (torch.randn(E, 2 * F, H, generator=g, device=DEV) * H ** -0.5).to(torch.bfloat16)
    down = (torch.randn(E, H, F, generator=g, device=DEV) * F ** -0.5).to(torch.bfloat16)
    w = torch.rand(n, top, generator=g, device=DEV)
    act, y = (torch.full((n, top, k), 7.0, dtype=torch.bfloat16, device=DEV) for k in (F, H))
    out = torch.empty(n, H, device=DEV)
    names = launched.kernels(lambda: call(E, n, h, up, down, idx, w, act, y, out, True, "silu"))
    assert sum("moe_product" in x for x in names) == 2
    idle = idx >= E
    assert 0 < int(idle.sum()) < n * top and bool((act[idle] == 7).all()) and bool((y[idle] == 7).all())
    want = torch.zeros(n, H, dtype=torch.float64, device=DEV)
    flat, size = idx.flatten(), torch.zeros(n, H, dtype=torch.float64, device=DEV)
    for e in range(E + 8):
        mine = (flat == e).nonzero()[:, 0]
        t, k = mine // top, mine % top
        x = h[t].double()
        if e < E:
            z = x @ up[e].double().T
            a = torch.nn.functional.silu(z[:, :F]) * z[:, F:]
            v, s = a @ down[e].double().T, a.abs() @ down[e].double().abs().T
            # act is rounded to 8 bits, 2^-8 of itself, its float sums of 2,048 and the result's of 1,728 numbers to 2^-12 of their sizes, y to 2^-8
            off = (2.0 ** -8 + 2.0 ** -12) * s + 2.0 ** -8 * v.abs()
        else:
            v, off = x, torch.zeros_like(x)
        want.index_add_(0, t, w[t, k, None].double() * v)
        size.index_add_(0, t, w[t, k, None].double() * off + 2.0 ** -20 * v.abs())
    assert bool(((out.double() - want).abs() <= size).all())
