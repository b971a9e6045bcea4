"""Decode steps over few keys: one share of a token's keys up to the sizes where a merge of several becomes cheaper."""
from types import SimpleNamespace

import pytest
import torch

from test_kernels_gpu import DEV, attention_reference, paged_setup, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,hd,most,shares", [(16, 2, 64, 767, 1), (16, 2, 64, 768, 6), (32, 2, 128, 511, 1), (32, 2, 128, 512, 4)])
def test_shares_of_few_keys(nh, nkv, hd, most, shares):
    from cpmcu_amd import ops
    lens, page, asked = (most, 1, 33), 64, []
    ks, vs, kpool, vpool, table = paged_setup(list(lens), nkv, hd, page, torch.bfloat16, seed=6)

    def get(name, shape, dtype):
        asked.append(shape)
        return torch.empty(shape, dtype=dtype, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(single_token=True, max_pos=most - 1, positions=i32([q - 1 for q in lens]), tok_slot=i32([0, 1, 2]),
                          ws=SimpleNamespace(get=get))
    q = rnd(len(lens), nh, hd, seed=7, dtype=torch.bfloat16)
    out = torch.empty(len(lens), nh * hd, dtype=torch.bfloat16, device=DEV)
    ops.attention(q.view(len(lens), -1), out, nh, nkv, hd, hd ** -0.5, kpool, vpool, table, page, ctx)
    assert [s[2] for s in asked] == ([shares] * 2 if shares > 1 else [])
    ref = attention_reference(q.double().cpu(), ks, vs, [n - 1 for n in lens], [0, 1, 2], nh, hd ** -0.5)
    top = max(float(v.abs().max()) for v in vs)            # weights and output are each rounded to 8 bits
    assert float((out.double().cpu().view(len(lens), nh, hd) - ref).abs().max()) <= 2 ** -8 * top
