"""Products head by head in tiles of 128: rows, columns and features that end inside a tile or a piece, slices of wider rows
that do and do not allow joint writes, both kinds of gate (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,M,N,K", [(256, 17, 8, 8), (64, 130, 129, 72), (128, 129, 6, 128), (32, 1024, 132, 64), (256, 128, 127, 200),
                                     # in tiles of 128: full ones, whose last columns or features end inside a piece ...
                                     (256, 65, 72, 72), (16, 2000, 127, 64), (128, 128, 250, 136),
                                     # ... three quarters, half and fewer, and beside each what stays in tiles of 64
                                     (64, 130, 510, 128), (32, 130, 510, 128), (64, 300, 131, 280), (128, 129, 67, 264), (256, 24, 128, 256),
                                     (256, 23, 128, 256), (256, 64, 64, 256)])
@pytest.mark.parametrize("gate", [None, "head", "feature"])
@pytest.mark.parametrize("odd", [False, True])
def test_head_products_at_tile_edges(H, M, N, K, gate, odd):
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(H + M + N + K)
    xs, ys, pad = K + 8, N + (3 if odd else -N % 4), 1 if odd else 4
    x = torch.randn(M, 16 + H * xs, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(H, N, K, generator=g, device=DEV).to(torch.bfloat16)
    out = torch.full((M, pad + H * ys), float("nan"), dtype=torch.bfloat16, device=DEV)
    gates = None if gate is None else torch.randn(M, H * (N if gate == "feature" else 1), generator=g, device=DEV).to(torch.bfloat16)
    ops.gemm_heads(x, 16, xs, w, out, pad, ys, gate=gates)
    xh = x[:, 16:].view(M, H, xs)[:, :, :K].permute(1, 0, 2).double()
    ref, mag = torch.matmul(xh, w.double().transpose(1, 2).contiguous()), torch.matmul(xh.abs(), w.double().abs().transpose(1, 2).contiguous())
    got = out[:, pad:].view(M, H, ys).permute(1, 0, 2)
    if gates is not None:
        s = torch.sigmoid(gates.double().view(M, H, -1)).permute(1, 0, 2)
        ref, mag = ref * s, mag * s
    # float sums in any order (and an exponential), then one rounding to bf16
    assert bool(((got[..., :N].double() - ref).abs() <= (K + 8) * 2.0 ** -23 * mag + 2.0 ** -8 * ref.abs()).all())
    assert bool(torch.isnan(out[:, :pad]).all()) and bool(torch.isnan(got[..., N:]).all())        # nothing written beside
