"""Gated experts of few tokens: tokens that share an expert are taken together, several runs of pairs, identity experts."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,top,E,H,F", [(1, 2, 4, 64, 32), (9, 3, 3, 72, 19), (13, 2, 7, 520, 33), (70, 3, 5, 36, 18), (129, 1, 2, 8, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_shared_experts_like_lone_ones(n, top, E, H, F, dtype):
    from cpmcu_amd import ops
    g = torch.Generator().manual_seed(n + E)
    # the highest number is an identity expert: nothing may be written for it
    idx = torch.stack([torch.randperm(E + 1, generator=g)[:top] for _ in range(n)]).to(torch.int32)
    h = torch.randn(n, H, generator=g).to(dtype)
    gu = (torch.randn(E, 2 * F, H, generator=g) * H ** -0.5).to(dtype)
    act = torch.full((n, top, F), float("nan"), dtype=dtype, device=DEV)
    ops.moe_gated(h.to(DEV), gu.to(DEV), idx.to(DEV), act)
    one = torch.full((n, top, F), float("nan"), dtype=dtype, device=DEV)
    for t in range(n):
        ops.moe_gated(h[t:t + 1].to(DEV), gu.to(DEV), idx[t:t + 1].to(DEV), one[t:t + 1])
    real = (idx < E).to(DEV)
    assert torch.equal(act[real], one[real]) and bool(act[~real].isnan().all())
    z = torch.einsum("nh,ejh->nej", h.double(), gu.double())
    gate, up = z[..., :F], z[..., F:]
    want = (torch.nn.functional.silu(gate) * up).gather(1, idx.clamp(max=E - 1).long()[..., None].expand(n, top, F))
    off = (act.double().cpu() - want)[idx < E].abs().max()
    # float sums over H of products of order 1 / sqrt(H), then one rounding to 8 bits
    assert float(off) <= (2 ** -8 if dtype == torch.bfloat16 else 1e-5) * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("n,top", [(3, 6), (9, 2), (50, 3), (2, 16)])
@pytest.mark.parametrize("H,F", [(2052, 2056), (2048, 2048)])
@pytest.mark.parametrize("shared_dtype", [None, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("joined", [False, True])
def test_down_rows_read_once_for_all_pairs(n, top, H, F, shared_dtype, joined):
    """Experts of 8 MiB and 18 pairs or more: rows by pair and a token's sum, beside a sum in double; lone and shared experts, up
    to four pairs at a time and more, more than one run of 128 pairs, identity experts; the same without scratch."""
    from cpmcu_amd import ops
    E = 4
    g = torch.Generator(device=DEV).manual_seed(n + H)
    rnd = lambda *shape, dtype=torch.bfloat16: torch.randn(*shape, generator=g, device=DEV).to(dtype)
    act, down, h = rnd(n, top, F), rnd(E, H, F, dtype=torch.bfloat16) * F ** -0.5, rnd(n, H)
    idx = torch.randint(0, E + 1, (n, top), generator=torch.Generator().manual_seed(n), dtype=torch.int32).to(DEV)
    w = torch.rand(n, top, generator=g, device=DEV)
    shared = None if shared_dtype is None else rnd(19, n, H, dtype=shared_dtype) if shared_dtype == torch.float32 else rnd(n, H)
    sg = None if shared is None else torch.rand(n, generator=g, device=DEV)
    x0, a, bias = rnd(n, H, dtype=torch.float32), rnd(18, n, H, dtype=torch.float32), rnd(H, dtype=torch.float32)
    assert n * top >= 18 and H * F >= 4 << 20

    def run(scratch):
        x, copy, out = x0.clone(), torch.empty(n, H, dtype=torch.bfloat16, device=DEV), torch.empty(n, H, device=DEV)
        join = ops.Join(x, a, bias, copy) if joined else None
        ops.moe_down(act, down, idx, w, None if joined else out, shared, sg, h=h, join=join, pair_out=scratch)
        return (x if joined else out), copy

    y = torch.full((n, top, H), float("nan"), device=DEV)
    (got, copy), (old, _) = run(y), run(None)
    real = idx < E
    assert torch.equal(y.isnan().any(-1), ~real) and torch.equal(y.isnan().all(-1), ~real)
    rows = h.double()[:, None].expand(n, top, H).clone()
    mags = rows.abs()
    for e in range(E):
        at = idx == e
        rows[at] = act[at].double() @ down[e].double().T
        mags[at] = act[at].double().abs() @ down[e].double().abs().T
    terms = [w.double()[..., None] * rows]
    mag = (w.double()[..., None] * mags * F).sum(1)                      # F products and their sums, in float
    if shared is not None:
        s = shared.double() if shared.dim() == 3 else shared.double()[None]
        terms.append((sg.double()[:, None] * s).transpose(0, 1))
    if joined:
        terms += [x0.double()[:, None], a.double().transpose(0, 1), bias.double().expand(n, H)[:, None]]
        assert torch.equal(copy, got.to(torch.bfloat16))
    terms = torch.cat(terms, 1)
    off = 2.0 ** -24 * (2 * mag + 2 * terms.shape[1] * terms.abs().sum(1))
    for t in (got, old):
        assert bool(((t.double() - terms.sum(1)).abs() <= off).all())
