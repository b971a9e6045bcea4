"""Products of decode steps by strips of output columns, at the borders of the rules that share their work out (GPU)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, g, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


@pytest.mark.parametrize("n,I,K", [(17, 16, 8), (32, 4096, 1024), (33, 48, 1000), (64, 1008, 136), (64, 16, 1024)])
@pytest.mark.parametrize("scaled", [False, True])
def test_gated_strips_of_up_to_64_tokens(n, I, K, scaled):
    from cpmcu_amd import ops
    assert ops.gated_strip_ok(n, K) and not ops.gated_strip_ok(n, 1032) and not ops.gated_strip_ok(65, 8)
    g = torch.Generator(device=DEV).manual_seed(n + K)
    x, w = rnd(n, K, g=g, dtype=torch.bfloat16), rnd(2 * I, K, g=g, dtype=torch.bfloat16, scale=2.0 * K ** -0.5)
    rs, r = None, 1.0
    if scaled:
        rs = ops.RowScale(torch.rand(n, 5, generator=g, device=DEV) + 0.1, 1e-3)
        r = torch.rsqrt(rs.sums.double().sum(1) / K + 1e-3).view(n, 1)
    out = torch.full((n, I), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gated_strip(x, ops.TiledWeight(w), out, row_scale=rs, most=64)
    y = (x.double() @ w.double().T) * r
    ref = F.silu(y[:, :I]) * y[:, I:]
    # the output's rounding, and K float sums of terms of order one before the nonlinearity
    assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4 * (1 + y[:, I:].abs())).all())
    with pytest.raises(ops.KernelError):
        ops.gated_strip(rnd(17, 1032, g=g, dtype=torch.bfloat16), ops.TiledWeight(rnd(32, 1032, g=g, dtype=torch.bfloat16)),
                        torch.empty(17, 16, dtype=torch.bfloat16, device=DEV), most=64)


@pytest.mark.parametrize("n", [1, 16, 20, 32])
@pytest.mark.parametrize("K", [8, 1016, 1024, 1032, 12280, 12288])
def test_residual_products_at_the_borders_of_the_wavefronts_shares(n, K):
    """Up to 1,024 columns, up to 12,288 and beyond: blocks shared by 4 or 8 wavefronts, some of which have none."""
    from cpmcu_amd import ops
    N = 36
    g = torch.Generator(device=DEV).manual_seed(n + K)
    a, w = rnd(n, K, g=g, dtype=torch.bfloat16), rnd(N, K, g=g, dtype=torch.bfloat16, scale=K ** -0.5)
    x0, nw = rnd(n, N, g=g), rnd(N, g=g)
    x, xw, sums = x0.clone(), torch.empty(n, N, dtype=torch.bfloat16, device=DEV), torch.empty(n, 3, device=DEV)
    ops.proj_add_norm(a, ops.TiledWeight(w), 0.6, x, nw, xw, sums)
    want = x0.double() + 0.6 * (a.double() @ w.double().T)
    assert float((x.double() - want).abs().max()) <= 1e-5 * float(want.abs().max())
    assert float((sums.double().sum(1) - (want ** 2).sum(1)).abs().max()) <= 1e-5 * float((want ** 2).sum(1).max())


@pytest.mark.parametrize("n,K", [(17, 1024), (33, 8), (33, 1024), (48, 1000), (49, 136), (64, 1024)])
def test_residual_products_that_every_wavefront_finishes(n, K):
    """Up to four tiles of 16 tokens, one a wavefront at the end: the last one full, or one token of it."""
    test_residual_products_at_the_borders_of_the_wavefronts_shares(n, K)


@pytest.mark.parametrize("n,N,K", [(1, 16, 128), (8, 100, 1152), (16, 8192, 256), (9, 2000, 384), (3, 9000, 640), (8, 33000, 128), (16, 40, 4096), (2, 9000, 1024), (8, 33000, 1152)])
@pytest.mark.parametrize("mode,dtype", [("plain", torch.float32), ("plain", torch.bfloat16), ("act", torch.bfloat16)])
def test_products_of_one_wavefront_a_strip(n, N, K, mode, dtype):
    """Fewer blocks than are asked for ahead, one more, many; columns that end inside a strip: the results of the product that
    stages its rows through LDS (which takes the weight as it stands in the checkpoint), to the last bit."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n + N)
    x, w = rnd(n, K, g=g, dtype=torch.bfloat16), rnd(N, K, g=g, dtype=torch.bfloat16, scale=K ** -0.5)
    for rs in (None, ops.RowScale(torch.rand(n, 21, generator=g, device=DEV) + 0.1, 1e-3)):
        outs = [torch.full((n, N), float("nan"), dtype=dtype, device=DEV) for _ in range(2)]
        for weight, out in zip((ops.TiledWeight(w), w), outs):
            kw = {"activation": "relu_squared"} if mode == "act" else {}
            ops.gemm_skinny(x, weight, out, 0.75, mode=mode, row_scale=rs, **kw)
        assert torch.equal(*outs)


@pytest.mark.parametrize("n,H", [(33, 1024), (48, 1000), (49, 136), (64, 1024), (64, 8), (64, 1032)])
@pytest.mark.parametrize("scaled", [False, True])
def test_fused_projection_of_many_tokens(n, H, scaled):
    """33 to 64 tokens: 8 wavefronts a workgroup up to 1,024 columns, tile t of the tokens finished by wavefront t."""
    from test_kernels_gpu import test_fused_projection_rotation_and_cache_write as check
    for nh, nkv, hd in ((3, 1, 16), (2, 2, 64)):
        check(n, nh, nkv, hd, H, True, scaled, None)


@pytest.mark.parametrize("n,ks,st", [(64, 32, 16), (40, 12, 4)])
def test_compressed_keys_of_many_tokens(n, ks, st):
    """A mean's keys of this step may come from several wavefronts."""
    from test_kernels_gpu import test_fused_projection_completes_compressed_keys as check
    check(n, ks, st, None)
