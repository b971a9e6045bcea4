"""Kernels of steps that bring one token a sequence, beside the kernels that bring any number: the same results to the last bit
(GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, g, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,dk,dv", [(3, 64, 128), (2, 128, 70), (5, 40, 64), (1, 256, 16), (2, 192, 129)])
def test_gated_linear_steps_do_not_depend_on_the_batch(H, dk, dv, dtype):
    """More than 512 (sequence, head) pairs take workgroups of 512 threads, fewer take 1,024: the same results."""
    from cpmcu_amd import ops
    B, R = 512 // H + 1, 6
    g = torch.Generator(device=DEV).manual_seed(dk)
    rows = rnd(B, 2 * H * dk + 2 * H * dv + R, g=g, dtype=dtype)
    up, bias, w = rnd(R, H * dk, g=g), rnd(H * dk, g=g), torch.rand(dv, generator=g, device=DEV) + 0.5
    start = rnd(B, H, dv, dk, g=g)
    start[3, 0, dv - 1, dk - 1] = float("inf")
    off = (0, H * dk, 2 * H * dk, 2 * H * dk + H * dv, 2 * H * dk + 2 * H * dv)

    def run(a, b):
        state, out = start[a:b].clone(), torch.empty(b - a, H * dv, dtype=dtype, device=DEV)
        ops.gla_step(rows[a:b], *off, up, bias, 4.0, w, 1e-5, state, out, i32(list(range(b - a + 1))), i32(list(range(b - a))), H, dk, dv, 0.3)
        return out, state

    out, state = run(0, B)
    for a, b in ((0, 7), (B - 5, B)):
        o, s = run(a, b)
        assert torch.equal(torch.nan_to_num(o, 77.0), torch.nan_to_num(out[a:b], 77.0)) and torch.equal(torch.nan_to_num(s, 77.0), torch.nan_to_num(state[a:b], 77.0))
