"""The 32-bit engine's kernels on the matrix cores, at the edges of their tiles and of the rules that choose them (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# up to 16 rows (and up to 32,768 outputs), tiles of 32, 64 and 128, each with columns that end inside a piece of 32 or 64
# and with rows that start off 16-byte borders (K % 4 != 0)
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (16, 33, 300), (5, 32768, 7), (16, 32769, 12), (17, 31, 68), (33, 64, 65),
                                   (1025, 2048, 36), (1030, 2049, 33), (2048, 4097, 20), (2049, 4096, 35)])
def test_float_product_at_tile_edges(M, N, K):
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm_nt_plain(x, w, out, 1.5)
    ref = 1.5 * (x.double() @ w.double().T)
    # K products and sums, each rounded once, in any order: at most K + 1 roundings of a sum of the magnitudes
    bound = (K + 2) * 2.0 ** -24 * 1.5 * (x.double().abs() @ w.double().abs().T)
    assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("nh,nkv,hd", [(17, 1, 16), (6, 2, 128), (4, 4, 80)])
def test_float_attention_ignores_what_lies_behind_the_token(nh, nkv, hd):
    """A token's page may hold anything behind it, infinities too; 1, 2, 4, 5 and 9 chunks of 32 keys for 4 wavefronts."""
    from cpmcu_amd import ops
    page, pages = 64, 5
    g = torch.Generator(device=DEV).manual_seed(hd)
    kpool = torch.randn(pages, page, nkv * hd, generator=g, device=DEV)
    vpool = torch.randn(pages, page, nkv * hd, generator=g, device=DEV)
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None].contiguous()
    # the pages' element order, read back: key slot and value places of token t32 of a chunk
    t = torch.arange(pages * page)
    d = torch.arange(hd)
    t32 = t % 32
    slot = (t32 // 8) * 4 + t32 % 4
    chunk = (t // 32)[:, None, None] * nkv * 32 * hd + (torch.arange(nkv) * 32 * hd)[None, :, None]
    kat = chunk + (((t32 // 4) % 2) * hd * 16 + slot * 8)[:, None, None] + ((d // 8) * 128 + d % 8)
    vat = chunk + ((t32 // 8) * 128 + t32 % 8)[:, None, None] + ((d // 16) * 512 + (d % 16) * 8)
    k, v = kpool.flatten().cpu()[kat], vpool.flatten().cpu()[vat]                      # [tokens, nkv, hd]
    for pos in (0, 31, 32, 100, 130, 263):
        q = torch.randn(1, nh, hd, generator=g, device=DEV)
        kp, vp = kpool.clone(), vpool.clone()
        kp.view(-1)[kat[pos + 1:].flatten().to(DEV)] = float("inf")
        vp.view(-1)[vat[pos + 1:].flatten().to(DEV)] = float("inf")
        out = torch.full((1, nh * hd), float("nan"), device=DEV)
        at = torch.tensor([pos], dtype=torch.int32, device=DEV)
        ops.attention_plain(q.view(1, -1), out, nh, nkv, hd, hd ** -0.5, kp, vp, table, page, at, torch.zeros_like(at))
        rep = lambda x: x[:pos + 1].double().repeat_interleave(nh // nkv, 1)
        w = torch.softmax(torch.einsum("hd,jhd->hj", q[0].double().cpu(), rep(k)) * hd ** -0.5, -1)
        ref = torch.einsum("hj,jhd->hd", w, rep(v))
        assert float((out.double().cpu().view(nh, hd) - ref).abs().max()) <= 2e-6, pos
