"""Masks that no kernel takes are refused whatever the positions of the step."""
from types import SimpleNamespace

import pytest
import torch

from cpmcu_amd import ops


@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("max_pos", [5, 500])
@pytest.mark.parametrize("mask", [{"chunk": 64, "window": 64}, {"chunk": -1}, {"window": -7}, {"window": 64, "keep_first": -2},
                                  {"chunk": 64, "keep_first": 3}])
def test_masks_are_checked_as_they_are_given(mask, max_pos, single):
    ctx = SimpleNamespace(single_token=single, max_pos=max_pos, q_lens=[1 if single else 300])
    n, nh, nkv, hd, page = ctx.q_lens[0], 4, 2, 64, 64
    q, out = torch.zeros(n, nh * hd, dtype=torch.bfloat16), torch.zeros(n, nh * hd, dtype=torch.bfloat16)
    pool = torch.zeros(8, page, nkv * hd, dtype=torch.bfloat16)
    with pytest.raises(ops.KernelError, match="mask"):
        ops.attention_any(q, out, nh, nkv, hd, hd, 0.125, pool, pool, None, page, ctx, **mask)
