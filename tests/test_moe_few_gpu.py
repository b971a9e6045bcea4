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
