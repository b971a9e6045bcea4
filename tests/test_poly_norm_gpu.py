"""PolyNorm of 16-bit rows in 16-byte pieces: widths around a thread's first, third and fourth piece, and the last it takes."""
import pytest
import torch

import plain_duvulix as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("F", [8, 4088, 4096, 4104, 12288, 12296, 16384, 16392, 4100])
@pytest.mark.parametrize("n", [1, 5])
def test_poly_norm_of_16_bit_rows(n, F):
    from cpmcu_amd import ops
    g = torch.Generator().manual_seed(F + n)
    z = (torch.randn(n, F, generator=g) * 1.5).to(torch.bfloat16)
    coef = torch.tensor([0.9, -0.6, 0.5, 0.2])
    out = torch.full((n, F), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.poly_norm(z.to(DEV), coef.to(DEV), 1e-5, out)
    want = plain.poly_norm(z.double(), coef.double(), 1e-5)
    # one rounding to 8 bits (2^-9 relative); the float sums are far below
    off = (out.double().cpu() - want).abs()
    assert bool((off <= 2.0 ** -8 * want.abs() + 1e-5).all()), float(off.max())
