"""Products of many rows: every tile's form at the edges of tiles, rounds and pieces, results inside a wider buffer (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (65, 8, 128), (130, 264, 128), (257, 72, 192), (300, 1032, 320), (33, 520, 1024), (512, 512, 512),
                                   (1040, 2048, 64), (1500, 6176, 192), (2048, 9256, 128), (4000, 9256, 64)])
@pytest.mark.parametrize("kind", ["plain", "gated"])
def test_every_tile(M, N, K, kind):
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K + 16, generator=g, device=DEV).to(torch.bfloat16)[:, 8:K + 8]            # rows apart, 16 bytes in
    w = torch.randn(N * (2 if kind == "gated" else 1), K, generator=g, device=DEV).to(torch.bfloat16)
    if M > 2:
        x[M // 2, 5] = float("nan")                                    # reaches its own row only
    z = x.double() @ w.double().t()
    off = K * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())   # float sums in any order
    if kind == "gated":
        a, u = z[:, :N], z[:, N:]
        want = torch.nn.functional.silu(a) * u
        # |silu'| <= 1.1; the exponential's argument is rounded to 2^-24 of itself (|a| e^-|a| < 0.4 of a gate's value), the rest to a few bits
        off = 1.1 * off[:, :N] * u.abs() + (a.abs() + off[:, :N]) * off[:, N:] + 16 * 2.0 ** -23 * (1 + a.abs()) * want.abs()
    else:
        want = z
    off = off + 2.0 ** -8 * (want.abs() + off) + 1e-30
    for tile in range(13):
        if kind == "gated" and tile >= 10:
            continue                                                   # tiles of 192 weight rows hold no whole gates
        wide = torch.full((M + 1, N + 8), 7.0, device=DEV, dtype=torch.bfloat16)
        out = wide[:M, :N]
        ops.product(x, w, out, kind, tile=tile)
        rows = torch.arange(M, device=DEV) != (M // 2 if M > 2 else -1)
        assert bool(((out.double() - want).abs() <= off)[rows].all()), tile
        assert M <= 2 or bool(out[M // 2].isnan().all())
        assert bool((wide[M] == 7).all()) and bool((wide[:, N:] == 7).all())


@pytest.mark.parametrize("activation", ["gelu_tanh", ("clamped_swish", 1.5)])
def test_gates(activation):
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(256, 128, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * 200, 128, generator=g, device=DEV) * 128 ** -0.5).to(torch.bfloat16)
    out = torch.empty(256, 200, device=DEV, dtype=torch.bfloat16)
    ops.product(x, w, out, "gated", activation)
    z = x.double() @ w.double().t()
    a, u = z[:, :200], z[:, 200:]
    if activation == "gelu_tanh":
        want = torch.nn.functional.gelu(a, approximate="tanh") * u
    else:
        a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5)
        want = a * torch.sigmoid(1.702 * a) * (u + 1)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all())      # sums of 128 numbers of order one


def test_what_is_refused():
    from cpmcu_amd import ops
    x, w = torch.zeros(300, 128, device=DEV, dtype=torch.bfloat16), torch.zeros(64, 128, device=DEV, dtype=torch.bfloat16)
    out = torch.empty(300, 64, device=DEV, dtype=torch.bfloat16)
    ops.product(x, w, out)
    for bad in [(x[:, :96], w[:, :96], out), (x[:, 4:68], w[:, :64].contiguous(), out), (x.t().contiguous().t(), w, out), (x.float(), w, out),
                (x, w[:60], out[:, :60]), (x, w, out[:, :32]), (x, w, out.float()), (x, w[:, :64], out)]:
        with pytest.raises(ops.KernelError):
            ops.product(*bad)
    with pytest.raises(ops.KernelError):
        ops.product(x, w, out, tile=13)
    with pytest.raises(ops.KernelError):
        ops.product(x, w, out[:, :32], "gated", tile=12)


@pytest.mark.parametrize("rows,columns,strided,outputs,ours", [
    (300, 128, False, 8192, False), (300, 72, False, 8192, False), (300, 128, True, 8192, False), (255, 128, False, 8192, False), (2048, 64, False, 8192, False),
    # where the rule names the kernel: operands that it takes, and others
    (300, 4096, False, 4096, True), (300, 4096, True, 4096, False), (300, 4104, False, 4096, False), (300, 4096, False, 4100, False),
    (1040, 128, False, 4096, True), (1040, 128, True, 4096, False), (1040, 136, False, 4096, False)])
def test_linear_takes_what_it_took(rows, columns, strided, outputs, ours):
    """The dispatcher's two ways for many rows, with operands that the kernel does not take among them."""
    from cpmcu_amd import ops
    import launched
    assert ops.product_faster(rows, outputs, columns) == (outputs < 8192)
    g = torch.Generator(device=DEV).manual_seed(rows + columns)
    x = torch.randn(rows, columns, generator=g, device=DEV).to(torch.bfloat16)
    if strided:
        x = x.t().contiguous().t()
    w = torch.randn(outputs, columns, generator=g, device=DEV).to(torch.bfloat16)
    out = torch.empty(rows, outputs, device=DEV, dtype=torch.bfloat16)
    assert any("product_kernel" in n for n in launched.kernels(lambda: ops.linear(x, w, out))) == ours
    want = x.double() @ w.double().t()
    off = columns * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())
    assert bool(((out.double() - want).abs() <= off + 2.0 ** -8 * (want.abs() + off)).all())


@pytest.mark.parametrize("M,N,K,parts", [(1, 8, 512, 2), (65, 264, 1024, 4), (130, 72, 768, 3), (257, 520, 512, 1), (300, 1032, 2048, 8), (704, 2056, 512, 2), (1500, 1032, 1024, 2)])
@pytest.mark.parametrize("activation", [None, "silu", ("clamped_swish", 1.5)])
def test_shares_of_the_columns(M, N, K, parts, activation):
    """Every tile; sums of shares in their order, results inside a wider buffer, a row that is no number."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = (torch.randn(M, K + 16, generator=g, device=DEV) * K ** -0.5).to(torch.bfloat16)[:, 8:K + 8]
    w = torch.randn(N * (2 if activation else 1), K, generator=g, device=DEV).to(torch.bfloat16)
    if M > 2:
        x[M // 2, 5] = float("nan")
    z = x.double() @ w.double().t()
    off = K * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())
    if activation:
        a, u, slack = z[:, :N], z[:, N:], 16 * 2.0 ** -23
        if activation != "silu":
            a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5) + 1
        want = a * torch.sigmoid(a if activation == "silu" else 1.702 * a) * u
        off = 1.1 * off[:, :N] * u.abs() + (a.abs() + off[:, :N]) * off[:, N:] + slack * (1 + 1.702 * a.abs()) * want.abs()
    else:
        want = z
    off = off + 2.0 ** -8 * (want.abs() + off) + 1e-30
    rows = torch.arange(M, device=DEV) != (M // 2 if M > 2 else -1)
    for tile in range(-1, 13):
        wide = torch.full((M + 1, N + 8), 7.0, device=DEV, dtype=torch.bfloat16)
        ops.product_parts(x, w, wide[:M, :N], parts, activation is not None, activation or "silu", tile=tile)
        out = wide[:M, :N]
        assert bool(((out.double() - want).abs() <= off)[rows].all()), tile
        assert M <= 2 or activation not in (None, "silu") or bool(out[M // 2].isnan().all())
        assert bool((wide[M] == 7).all()) and bool((wide[:, N:] == 7).all())


def test_what_shares_refuse():
    from cpmcu_amd import ops
    x, w = torch.zeros(100, 1024, device=DEV, dtype=torch.bfloat16), torch.zeros(64, 1024, device=DEV, dtype=torch.bfloat16)
    out = torch.empty(100, 64, device=DEV, dtype=torch.bfloat16)
    ops.product_parts(x, w, out, 4)
    for bad in [(x, w, out, 3), (x, w, out, 8), (x, w, out, 0), (x, w, out.float(), 2), (x[:, :96], w[:, :96], out, 1)]:
        with pytest.raises(ops.KernelError):
            ops.product_parts(*bad)


@pytest.mark.parametrize("rows,outputs,columns,want", [(64, 4096, 4096, None), (65, 4096, 4096, "sum"), (704, 4096, 16384, "sum"), (705, 4096, 4096, "product"),
                                                       (65, 2808, 4096, None), (65, 2816, 4096, "sum"), (200, 16384, 4096, "product"), (300, 4096, 4104, None),
                                                       (192, 2816, 4096, "sum"), (193, 2816, 4096, None), (128, 8192, 4096, None), (129, 8192, 4096, "sum"),
                                                       (768, 4096, 16384, "sum"), (1500, 4096, 16384, "sum"), (2048, 4096, 16384, "product"),
                                                       (1406, 2048, 4096, None), (1407, 2048, 4096, "product"), (1040, 2048, 8192, "sum"),
                                                       (2100, 1024, 4096, None), (2100, 1032, 4096, "sum"), (1024, 16384, 256, None)])
def test_the_rule_of_many_rows(rows, outputs, columns, want):
    from cpmcu_amd import ops
    import launched
    x, w = torch.randn(rows, columns, device=DEV).to(torch.bfloat16), torch.randn(outputs, columns, device=DEV).to(torch.bfloat16)
    out = torch.empty(rows, outputs, device=DEV, dtype=torch.bfloat16)
    names = launched.kernels(lambda: ops.linear(x, w, out))
    assert any("product_kernel" in n for n in names) == (want is not None) and any("product_sum" in n for n in names) == (want == "sum")
    z, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    off = columns * 2.0 ** -23 * size
    assert bool(((out.double() - z).abs() <= off + 2.0 ** -8 * (z.abs() + off)).all())


def test_shares_inside_a_captured_graph():
    from cpmcu_amd import ops
    x, w = torch.randn(100, 4096, device=DEV).to(torch.bfloat16), torch.randn(4096, 4096, device=DEV).to(torch.bfloat16)
    out = torch.empty(100, 4096, device=DEV, dtype=torch.bfloat16)
    ops.linear(x, w, out)
    want = out.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.linear(x, w, out)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("rows,half,columns,want", [
    (65, 1408, 4096, "sum"), (300, 2816, 4096, "sum"), (700, 2816, 4096, "product"), (96, 8192, 2048, "product"), (2048, 1024, 192, "product"),
    (1500, 2048, 8192, "product"), (1024, 8192, 256, "library"), (300, 1400, 4096, "library"), (300, 2820, 4096, "halves"), (300, 2816, 4104, "library")])
@pytest.mark.parametrize("activation", ["silu", ("clamped_swish", 1.5)])
def test_gated_layers_of_many_rows(rows, half, columns, want, activation):
    """The layer's ways: the gate on the product's float sums, whole or of shares, or behind the library's product (or the kernel's, of halves
    that are no whole groups of 8 outputs)."""
    import types
    import launched
    from cpmcu_amd.parts.base import Runtime, Workspace
    from cpmcu_amd.parts.linear import Linear
    ws = Workspace(DEV)
    g = torch.Generator(device=DEV).manual_seed(rows + half)
    x = (torch.randn(rows, columns, generator=g, device=DEV) * columns ** -0.5).to(torch.bfloat16)
    weights = {k: torch.randn(half, columns, generator=g, device=DEV).to(torch.bfloat16) for k in ("gate", "up")}
    layer = Linear([("gate", half), ("up", half)], columns)
    layer.bind(weights, Runtime(torch.device(DEV), torch.bfloat16, ws, 4096, tiled_weights=False))
    ctx, out = types.SimpleNamespace(ws=ws), []
    names = launched.kernels(lambda: out.append(layer.forward_gated(x, ctx, "gu", activation=activation)))
    assert any("product_kernel" in n for n in names) == (want != "library") and any("silu" in n for n in names) == (want in ("library", "halves"))
    assert want == "halves" or any("product_sum" in n for n in names) == (want == "sum")
    z = torch.cat([x.double() @ weights[k].double().t() for k in ("gate", "up")], 1)
    off = columns * 2.0 ** -23 * torch.cat([x.double().abs() @ weights[k].double().abs().t() for k in ("gate", "up")], 1)
    if want in ("library", "halves"):
        off = off + 2.0 ** -8 * (z.abs() + off)                        # both halves are rounded to 8 bits
    a, u = z[:, :half], z[:, half:]
    if activation != "silu":
        a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5) + 1
    gate = a * torch.sigmoid(a if activation == "silu" else 1.702 * a)
    off = 1.13 * off[:, :half] * u.abs() + (gate.abs() + 1.13 * off[:, :half]) * off[:, half:] + 16 * 2.0 ** -23 * (1 + 1.702 * a.abs()) * (gate * u).abs()
    off = off + 2.0 ** -8 * ((gate * u).abs() + off) + 1e-30
    assert bool(((out[-1].double() - gate * u).abs() <= off).all())
