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


# every tile that the rule chooses (its workgroups up to 256: 32 x 32, 32 x 64, 80 x 32, 48 x 64, 64 x 64 with the columns shared
# out; beyond: 64 rows by 64, 128, 192 and 256), columns that end inside a piece of 32, rows on and off 16-byte borders
SPLITS = [(17, 40, 64), (130, 1000, 100), (260, 1100, 72), (523, 1024, 96), (523, 1023, 65), (700, 1020, 68), (1000, 1000, 257),
          (1030, 1100, 131), (2000, 1500, 64), (2000, 2300, 97), (1999, 3101, 164)]


@pytest.mark.parametrize("M,N,K", SPLITS)
def test_float_product_in_three_parts(M, N, K):
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    x *= 2.0 ** torch.randint(-40, 40, (M, 1), generator=g, device=DEV)                # rows of all sizes
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm_nt_plain(x, w, out, 1.5)
    ref, mag = (1.5 * (a @ b.T) for a, b in ((x.double(), w.double()), (x.double().abs(), w.double().abs())))
    # sums as above, and the left out product of last parts: below 2^-30 of a product
    assert bool(((out.double() - ref).abs() <= ((K + 2) * 2.0 ** -24 + 2.0 ** -30) * mag).all())
    # the error on the whole: no larger than that of a float sum with a rounding every 32 columns and two of the result
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -24 * (K / 32 + 2) ** 0.5


@pytest.mark.parametrize("M,N,K", [(130, 300, 64), (523, 1024, 64), (700, 1020, 68), (1000, 1000, 257), (1999, 3101, 164)])
def test_float_product_of_few_columns_that_matter(M, N, K):
    """Rows of which one element is not zero: the product itself, rounded once."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.zeros(M, K, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    at = torch.randint(0, K, (M,), generator=g, device=DEV)
    x[torch.arange(M, device=DEV), at] = torch.randn(M, generator=g, device=DEV)
    out = torch.empty(M, N, device=DEV)
    ops.gemm_nt_plain(x, w, out, 1.0)
    off = (out.double() - x.double() @ w.double().T).abs() / (x.double() @ w.double().T).abs()
    # half a unit of the result, the cut sums of the smaller products (7 times 2^-23 of what ends below 2^-6), the one left out
    assert float(off.max()) <= 2.0 ** -24 * (1 + 7 * 2.0 ** -5 + 2.0 ** -6)
    # on the whole that of a rounding: an even error in a unit of 2^-24 to 2^-23 of the result, and an eighth of it for the cuts
    assert float((off ** 2).mean() ** 0.5) <= 2.0 ** -24 / 3 ** 0.5 * 1.125


@pytest.mark.parametrize("M,N,K", [(130, 1000, 1000), (523, 1024, 4096), (1999, 3101, 1028)])
def test_float_product_of_positive_numbers_has_no_lean(M, N, K):
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M)
    x, w = torch.rand(M, K, generator=g, device=DEV), torch.rand(N, K, generator=g, device=DEV)
    out = torch.empty(M, N, device=DEV)
    ops.gemm_nt_plain(x, w, out, 1.0)
    ref = x.double() @ w.double().T
    # roundings go either way; the smaller products' sums, 2^-6 of the result at most, are cut by 7 units of 2^-23 at most
    assert abs(float(((out.double() - ref) / ref).mean())) <= 7 * 2.0 ** -29


@pytest.mark.parametrize("M,N,K", [(70, 130, 96), (130, 1000, 100), (1030, 1100, 131), (1999, 3101, 164)])
@pytest.mark.parametrize("down,up", [(-118, 80), (-122, 60), (-125, 90), (-135, 100)])
@pytest.mark.parametrize("which", ["rows", "weights"])
def test_float_product_of_values_that_three_parts_do_not_hold(M, N, K, down, up, which):
    """Elements below 2^-110, whose last part is below the smallest bf16, against large ones: results of ordinary size."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    small, large = (x, w) if which == "rows" else (w, x)
    small[small.shape[0] // 2] *= 2.0 ** down
    small[-1, 3] *= 2.0 ** down
    large[:, ::2] *= 2.0 ** up
    out = torch.empty(M, N, device=DEV)
    ops.gemm_nt_plain(x, w, out, 1.0)
    ref, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert bool(((out.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * mag + K * 2.0 ** -126).all())


@pytest.mark.parametrize("N,K,rows", [(1000, 1028, (17, 33, 130, 300, 523, 1100)), (1024, 64, (17, 600, 2100)), (300, 257, (20, 64, 4000)),
                                      (8192, 320, (40, 130, 700)), (33000, 96, (1, 16, 17, 32, 33, 100))])
def test_float_rows_do_not_depend_on_the_others(N, K, rows):
    """Beyond 16 rows (or 32,768 outputs) a row's result is the same to the last bit whatever tile the rule takes, beside
    infinities, NaNs and very small numbers too."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x, w = torch.randn(max(rows), K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    x[0, 5], x[7, 0], x[16, K - 1] = float("inf"), float("nan"), 2.0 ** -130
    x[20 % max(rows)] *= 2.0 ** -90
    w[13, 1], w[200, 2] = float("-inf"), 2.0 ** -125
    out = []
    for n in rows:
        y = torch.full((n, N), 7.0, device=DEV)
        ops.gemm_nt_plain(x[:n].contiguous(), w, y, 1.0)
        out.append(y.view(torch.int32))
    for y in out[:-1]:
        assert torch.equal(y, out[-1][:y.shape[0]])


@pytest.mark.parametrize("M,N,K", [(70, 130, 96), (1030, 1100, 131)])
def test_float_product_of_odd_values(M, N, K):
    """Infinities, NaNs, the largest floats and floats whose last parts no bf16 holds: the float instruction's results."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    for t, (row, value) in enumerate([(0, float("inf")), (17, float("-inf")), (33, float("nan")), (34, 3.4e38), (69, -torch.finfo(torch.float32).max)]):
        x[row, 7 * t] = value
    w[5, 3], w[100, K - 1] = float("inf"), float("nan")
    x[40] *= 2.0 ** -122
    x[41] *= 2.0 ** -100
    out = torch.full((M, N), 7.0, device=DEV)
    ops.gemm_nt_plain(x, w, out, 1.0)
    ref = x.double() @ w.double().T
    mag = x.double().abs() @ w.double().abs().T
    fine = torch.isfinite(ref) & (mag < 1e38)
    assert torch.equal(out.isnan(), ref.isnan())
    assert bool((out.double() == ref)[torch.isinf(ref)].all())
    # (denormal products may be flushed one by one)
    assert bool(((out.double() - ref).abs() <= ((K + 2) * 2.0 ** -24 + 2.0 ** -30) * mag + K * 2.0 ** -126)[fine].all())
    assert bool(((out[40].double() - ref[40]).abs() <= (K + 2) * 2.0 ** -24 * mag[40] + K * 2.0 ** -126)[fine[40]].all())


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


def test_float_product_of_rows_far_apart():
    """Rows 2^28 floats apart: the last of 17 lies beyond what 32-bit offsets reach."""
    from cpmcu_amd import ops
    M, N, K, ld = 17, 40, 128, 2 ** 28
    g = torch.Generator(device=DEV).manual_seed(1)
    rows, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    x = torch.empty((M - 1) * ld + K, device=DEV).as_strided((M, K), (ld, 1))
    x.copy_(rows)
    out, want = torch.full((M, N), float("nan"), device=DEV), torch.empty(M, N, device=DEV)
    ops.gemm_nt_plain(rows, w, want, 1.0)
    ops._check(ops._fn("gemm", "cpmcu_gemm_nt_plain")(ops._p(x), ops.c_long(ld), ops._p(w), ops.c_long(K), ops._p(out), ops.c_long(N),
                                                      ops.c_int(ops._code(x)), ops.c_int(ops._code(out)), ops.c_int(M), ops.c_int(N),
                                                      ops.c_int(K), ops.c_float(1.0), ops._stream()))
    assert torch.equal(out, want)
