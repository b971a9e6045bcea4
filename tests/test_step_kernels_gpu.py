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


@pytest.mark.parametrize("lanes", [0, 8, 16])
@pytest.mark.parametrize("rule", ["channel", "decay", "delta"])
@pytest.mark.parametrize("B,H,kv,dk,dv", [(1, 4, 2, 128, 128), (5, 3, 1, 40, 33), (9, 2, 2, 200, 70), (3, 5, 5, 7, 9), (2, 2, 1, 256, 16)])
def test_delta_steps_beside_the_walk(B, H, kv, dk, dv, rule, lanes):
    """A sequence of two tokens more and the step's kernel gives way to the walk: the other sequences' results are the same
    (with one decay a head, whose products the compiler may fuse either way: to a rounding of either term)."""
    from cpmcu_amd import ops
    kv = H if rule == "decay" else kv
    g = torch.Generator(device=DEV).manual_seed(B * dk)
    n = B + 2
    qkv, gates = rnd(n, 2 * kv * dk + H * dv, g=g), rnd(n, 2 * H, g=g, dtype=torch.bfloat16)
    A = torch.rand(H, generator=g, device=DEV)
    bias = None if rule == "decay" else rnd(H * dk if rule == "channel" else H, g=g)
    decay = rnd(n, H * dk, g=g) if rule == "channel" else None
    start = rnd(B + 1, H, dv, dk, g=g)
    start[0, 0, dv - 1, dk - 1] = float("inf")
    scale = dk ** -0.5

    def run(rows, cu):
        state, y = start.clone(), torch.full((rows, H * dv), float("nan"), device=DEV)
        ops.delta_scan(qkv[:rows], None if rule == "decay" else gates[:rows], 0, H, bias, A, state, y, i32(cu), i32(list(range(len(cu) - 1))),
                       H, kv, dk, dv, scale, rule=rule, channel_decay=None if decay is None else decay[:rows], lanes=lanes)
        return y, state

    y, state = run(B, list(range(B + 1)))
    wy, wstate = run(n, list(range(B + 1)) + [n])
    wy, wstate = wy[:B], wstate[:B]
    assert torch.equal(state[B:], start[B:])
    state = state[:B]
    if rule != "delta":
        assert torch.equal(torch.nan_to_num(y, 77.0), torch.nan_to_num(wy, 77.0)) and torch.equal(torch.nan_to_num(state, 77.0), torch.nan_to_num(wstate, 77.0))
        return
    ulp = 2.0 ** -23
    ok = wstate.isfinite()
    assert bool((ok == state.isfinite()).all())
    assert bool((((state - wstate).abs() <= ulp * (2 * start[:B].abs() + wstate.abs()) + 1e-30) | ~ok).all())
    norm, v = start[:B].norm(dim=-1), qkv[:B, 2 * kv * dk:].view(B, H, dv).abs()
    ok = wy.isfinite()
    assert bool((ok == y.isfinite()).all())
    assert bool((((y - wy).abs() <= (ulp * scale * (2 * norm + v)).view(B, H * dv)) | ~ok).all())
