"""Recurrences taken 64 tokens at a time against a walk in double: runs that end inside, at and behind a chunk, several
sequences, a state that is carried on, sizes that do not fill a tile (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def off(got, want):
    return float((got.double().cpu() - want).norm() / want.norm())


@pytest.mark.parametrize("H,P,N,G,scale", [(4, 64, 128, 2, 1.0), (3, 36, 20, 1, 1.0), (2, 8, 64, 2, 6.0), (1, 4, 4, 1, 0.05)])
def test_state_space_chunks(H, P, N, G, scale):
    """`scale` stretches the step sizes: strong decays within a chunk, and nearly none."""
    from cpmcu_amd import ops
    g = torch.Generator().manual_seed(P + N)
    first, second = [17, 64, 65, 200], [64, 1, 130, 16]
    width = H * P + 2 * G * N
    A_log, bias, D = torch.log(0.05 + 3 * torch.rand(H, generator=g)), torch.randn(H, generator=g), torch.randn(H, generator=g)
    state = torch.zeros(6, H, P, N, device=DEV)
    walked = state.clone()
    S = [torch.zeros(H, P, N, dtype=torch.float64) for _ in first]
    slots = [4, 0, 5, 2]
    for lens in (first, second):
        n = sum(lens)
        cu = [0]
        for q in lens:
            cu.append(cu[-1] + q)
        xbc, dt = torch.randn(n, width, generator=g), torch.randn(n, H, generator=g) * scale
        want = torch.empty(n, H, P, dtype=torch.float64)
        d = torch.nn.functional.softplus(dt.double() + bias.double())
        x = xbc[:, :H * P].double().view(n, H, P)
        B, C = (xbc[:, H * P + k * G * N:H * P + (k + 1) * G * N].double().view(n, G, N).repeat_interleave(H // G, 1) for k in (0, 1))
        for s, q in enumerate(lens):
            for t in range(cu[s], cu[s] + q):
                S[s] = torch.exp(-torch.exp(A_log.double()) * d[t])[:, None, None] * S[s] + (d[t][:, None] * x[t])[:, :, None] * B[t][:, None]
                want[t] = (S[s] * C[t][:, None]).sum(-1) + D.double()[:, None] * x[t]
        outs = []
        for st, most in ((state, max(lens)), (walked, 0)):
            y = torch.full((n, H * P), float("nan"), device=DEV)
            ops.ssm_scan(xbc.to(DEV), dt.to(DEV), bias.to(DEV), A_log.to(DEV), D.to(DEV), st, y, i32(cu), i32(slots), H, P, N, G, max_q=most)
            outs.append(off(y.view(n, H, P), want))
        final = torch.stack(S)
        here, walk = (off(st[slots], final) for st in (state, walked))
        # float sums of up to 64 + N terms, every factor an exponential good to an ulp or two
        assert outs[0] <= 2e-6 and here <= 2e-6, (outs, here, walk)
        assert outs[0] <= 1.5 * outs[1] + 2e-7 and here <= 1.5 * walk + 2e-7, (outs, here, walk)
    assert float(state[[1, 3]].abs().max()) == 0.0


@pytest.mark.parametrize("H,G,dk,dv,scale", [(4, 2, 128, 128, 1.0), (3, 3, 36, 20, 1.0), (2, 1, 64, 40, 8.0), (2, 2, 4, 4, 0.05)])
def test_delta_rule_chunks(H, G, dk, dv, scale):
    """`scale` stretches decay and write rates.  Keys share a direction, so that the triangular system is far from the
    identity."""
    from cpmcu_amd import ops
    g = torch.Generator().manual_seed(dk + dv)
    first, second = [17, 64, 65, 200], [64, 1, 130, 16]
    A_log, bias = torch.log(0.05 + 3 * torch.rand(H, generator=g)), torch.randn(H, generator=g)
    state = torch.zeros(6, H, dv, dk, device=DEV)
    walked = state.clone()
    S = torch.zeros(4, H, dv, dk, dtype=torch.float64)
    slots, rep = [4, 0, 5, 2], H // G
    for lens in (first, second):
        n, cu = sum(lens), [0]
        for q in lens:
            cu.append(cu[-1] + q)
        qkv, gates = torch.randn(n, 2 * G * dk + H * dv, generator=g), torch.randn(n, 2 * H + 1, generator=g) * scale
        qkv[:, G * dk:2 * G * dk] += 1.0
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        Q = unit(qkv[:, :G * dk].double().view(n, G, dk)).repeat_interleave(rep, 1) * dk ** -0.5
        K = unit(qkv[:, G * dk:2 * G * dk].double().view(n, G, dk)).repeat_interleave(rep, 1)
        V = qkv[:, 2 * G * dk:].double().view(n, H, dv)
        keep = torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(gates[:, 1:1 + H].double() + bias.double()))
        beta = torch.sigmoid(gates[:, 1 + H:].double())
        want = torch.empty(n, H, dv, dtype=torch.float64)
        for s in range(4):
            for t in range(cu[s], cu[s + 1]):
                S[s] *= keep[t][:, None, None]
                u = beta[t][:, None] * (V[t] - (S[s] * K[t][:, None]).sum(-1))
                S[s] += u[:, :, None] * K[t][:, None]
                want[t] = (S[s] * Q[t][:, None]).sum(-1)
        outs = []
        for st, most in ((state, max(lens)), (walked, 0)):
            y = torch.full((n, H * dv), float("nan"), device=DEV)
            ops.delta_scan(qkv.to(DEV), gates.to(DEV), 1, 1 + H, bias.to(DEV), A_log.to(DEV), st, y, i32(cu), i32(slots), H, G, dk, dv,
                           dk ** -0.5, max_q=most)
            outs.append(off(y.view(n, H, dv), want))
        here, walk = (off(st[slots], S) for st in (state, walked))
        assert outs[0] <= 5e-6 and here <= 5e-6, (outs, here, walk)
        assert outs[0] <= 1.5 * outs[1] + 2e-7 and here <= 1.5 * walk + 2e-7, (outs, here, walk)
    assert float(state[[1, 3]].abs().max()) == 0.0


@pytest.mark.parametrize("H,d,dv,scale", [(2, 256, 64, 1.0), (3, 128, 32, 8.0), (2, 36, 20, 1.0), (1, 4, 4, 0.05)])
def test_mlstm_chunks(H, d, dv, scale):
    """`scale` stretches the gates: the running maximum then jumps within a chunk, or hardly moves."""
    from cpmcu_amd import ops
    g = torch.Generator().manual_seed(d + dv)
    first, second, cap = [17, 32, 33, 150], [64, 1, 65, 16], 15.0
    ib, fb = torch.randn(H, generator=g), torch.randn(H, generator=g) + 2.0
    zeros = lambda *s: torch.zeros(*s, device=DEV)
    states = [(zeros(6, H, dv, d), zeros(6, H, d), zeros(6, H)) for _ in range(2)]
    S, N, M = (torch.zeros(4, *s, dtype=torch.float64) for s in ((H, dv, d), (H, d), (H,)))
    slots, ko, vo, io, fo = [4, 0, 5, 2], H * d, 2 * H * d, 2 * H * d + H * dv, 2 * H * d + H * dv + H
    for lens in (first, second):
        n, cu = sum(lens), [0]
        for q in lens:
            cu.append(cu[-1] + q)
        proj = torch.randn(n, -(-(fo + H) // 4) * 4, generator=g)
        proj[:, io:fo + H] *= scale
        Q, K = (proj[:, o:o + H * d].double().view(n, H, d) for o in (0, ko))
        V = proj[:, vo:vo + H * dv].double().view(n, H, dv)
        a = cap * torch.tanh((proj[:, io:io + H].double() + ib.double()) / cap)
        b = torch.nn.functional.logsigmoid(cap * torch.tanh((proj[:, fo:fo + H].double() + fb.double()) / cap))
        want = torch.empty(n, H, dv, dtype=torch.float64)
        for s in range(4):
            for t in range(cu[s], cu[s + 1]):
                new = torch.maximum(b[t] + M[s], a[t])
                keep, take = torch.exp(b[t] + M[s] - new)[:, None], torch.exp(a[t] - new)[:, None] * K[t]
                S[s], N[s], M[s] = keep[..., None] * S[s] + V[t][:, :, None] * take[:, None], keep * N[s] + take, new
                qt = Q[t] * d ** -0.5
                low = torch.maximum((N[s] * qt).sum(-1).abs(), torch.exp(-new)) + 1e-6
                want[t] = (S[s] * qt[:, None]).sum(-1) / low[:, None]
        errs = []
        for (st, ns, ms), most in zip(states, (max(lens), 0)):
            y, den = torch.full((n, H * dv), float("nan"), device=DEV), torch.full((n, H), float("nan"), device=DEV)
            ops.mlstm_scan(proj.to(DEV), 0, ko, vo, io, fo, ib.to(DEV), fb.to(DEV), cap, d ** -0.5, st, ns, ms, y, den, i32(cu),
                           i32(slots), H, d, dv, max_q=most)
            scale_out = torch.exp(ms[slots].double().cpu() - M)            # a maximum a rounding away scales S and n alike
            errs.append([off(y.view(n, H, dv) / den[..., None], want), off(st[slots].double().cpu() * scale_out[..., None, None], S),
                         off(ns[slots].double().cpu() * scale_out[..., None], N), float((ms[slots].double().cpu() - M).abs().max())])
        assert all(h <= 1.5 * w + 5e-7 for h, w in zip(*errs)), errs
        assert errs[0][1] <= 2e-6 and errs[0][2] <= 2e-6, errs
    assert all(float(t[[1, 3]].abs().max()) == 0.0 for t in states[0])


# 64 sequences a ballot: the last one chosen alone, on both sides of that border, all in turn; every one of them or none
@pytest.mark.parametrize("kind", ["ssm", "delta", "mlstm"])
@pytest.mark.parametrize("lens,chunk_from", [([64, 1, 17, 130, 3], 64), ([1] * 63 + [33, 70, 1, 40], 40), ([5, 70] * 34, 70), ([9, 40], 9),
                                             ([66, 2], 67)])
def test_runs_are_taken_by_their_length(kind, lens, chunk_from):
    """Long runs in chunks, short ones walked, in one call: every run as in a call of its own form, bit by bit."""
    from cpmcu_amd import ops
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    B, n, cu = len(lens), sum(lens), [0]
    for q in lens:
        cu.append(cu[-1] + q)
    H, slots = 2, torch.randperm(B + 1, generator=torch.Generator().manual_seed(B))[:B].tolist()
    if kind == "ssm":
        P, N, states = 36, 20, [rnd(B + 1, H, 36, 20)]
        xbc, dt, A, b, D = rnd(n, H * P + 2 * N), rnd(n, H), rnd(H), rnd(H), rnd(H)
        call = lambda y, st, **k: ops.ssm_scan(xbc, dt, b, A, D, st[0], y[0], i32(cu), i32(slots), H, P, N, 1, **k)
        outs = [(n, H * P)]
    elif kind == "delta":
        dk, dv, states = 36, 20, [rnd(B + 1, H, 20, 36)]
        qkv, gates, A, b = rnd(n, 2 * H * dk + H * dv), rnd(n, 2 * H), rnd(H), rnd(H)
        call = lambda y, st, **k: ops.delta_scan(qkv, gates, 0, H, b, A, st[0], y[0], i32(cu), i32(slots), H, H, dk, dv, dk ** -0.5, **k)
        outs = [(n, H * dv)]
    else:
        d, dv, states = 36, 20, [rnd(B + 1, H, 20, 36), rnd(B + 1, H, 36), rnd(B + 1, H)]
        w = 2 * H * d + H * dv
        proj, b = rnd(n, w + 2 * H), rnd(H)
        call = lambda y, st, **k: ops.mlstm_scan(proj, 0, H * d, 2 * H * d, w, w + H, b, b, 9.0, d ** -0.5, *st, *y, i32(cu), i32(slots),
                                                 H, d, dv, **k)
        outs = [(n, H * dv), (n, H)]
    got = []
    chosen = [q >= chunk_from for q in lens]
    for k in (dict(chunks=(chunk_from, sum(chosen))), dict(chunks=(1, B)), dict(max_q=0)):
        y, st = [torch.full(o, float("nan"), device=DEV) for o in outs], [s.clone() for s in states]
        call(y, st, **k)
        got.append((y, st))
    both, chunked, walked = got
    for s in range(B):
        like = chunked if chosen[s] else walked
        assert all(torch.equal(a[cu[s]:cu[s + 1]], b[cu[s]:cu[s + 1]]) for a, b in zip(both[0], like[0])), s
        assert all(torch.equal(a[slots[s]], b[slots[s]]) for a, b in zip(both[1], like[1])), s
    left = next(i for i in range(B + 1) if i not in slots)
    assert all(torch.equal(a[left], b[left]) for a, b in zip(both[1], states))
    assert all(bool(torch.isfinite(y).all()) for y in both[0])


ODD = [("value", float("inf")), ("value", float("nan")), ("key", float("-inf")), ("key", float("nan")), ("query", float("inf")),
       ("gate", float("nan")), ("gate", float("inf")), ("gate", float("-inf")), ("second gate", float("nan")), ("constant", 100.0),
       ("constant", float("nan"))]


@pytest.mark.parametrize("kind", ["ssm", "delta", "mlstm"])
@pytest.mark.parametrize("what,odd", ODD)
@pytest.mark.parametrize("at", [5, 77, 90, 130])
def test_an_odd_token_reaches_what_the_walk_says(kind, what, odd, at):
    """An infinity or a NaN (or a decay constant whose exponential is infinite) in one token of a prompt: the same outputs and
    state values are finite as in the walk, and those have the walk's values; tokens before it see nothing of it, whether they
    stand in its block of 16 tokens, in its chunk, or before; the last token among them, behind which a chunk's rest is empty."""
    from cpmcu_amd import ops
    n, H = 131, 2
    g = torch.Generator(device=DEV).manual_seed(at)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    cu, slots = i32([0, n]), i32([1])
    if kind == "ssm":
        P, N, states = 36, 20, [rnd(2, H, 36, 20)]
        xbc, dt, A, b, D = rnd(n, H * P + 2 * N), rnd(n, H), torch.log(0.05 + rnd(H).abs()), rnd(H), rnd(H)
        place = {"value": (xbc, P + 3), "key": (xbc, H * P + 2), "query": (xbc, H * P + N + 7), "gate": (dt, 1)}
        call = lambda y, st, m: ops.ssm_scan(xbc, dt, b, A, D, st[0], y[0], cu, slots, H, P, N, 1, max_q=m)
        outs, constant = [(n, H, P)], A
    elif kind == "delta":
        dk, dv, states = 36, 20, [rnd(2, H, 20, 36)]
        qkv, gates, A, b = rnd(n, 2 * H * dk + H * dv), rnd(n, 2 * H), torch.log(0.05 + rnd(H).abs()), rnd(H)
        place = {"value": (qkv, 2 * H * dk + dv + 3), "key": (qkv, H * dk + dk + 2), "query": (qkv, dk + 7), "gate": (gates, 1),
                 "second gate": (gates, H + 1)}
        call = lambda y, st, m: ops.delta_scan(qkv, gates, 0, H, b, A, st[0], y[0], cu, slots, H, H, dk, dv, dk ** -0.5, max_q=m)
        outs, constant = [(n, H, dv)], A
    else:
        d, dv, states = 36, 20, [rnd(2, H, 20, 36), rnd(2, H, 36), rnd(2, H)]
        w = 2 * H * d + H * dv
        proj, b = rnd(n, w + 2 * H), rnd(H)
        place = {"value": (proj, 2 * H * d + dv + 3), "key": (proj, H * d + d + 2), "query": (proj, d + 7), "gate": (proj, w + 1),
                 "second gate": (proj, w + H + 1)}
        call = lambda y, st, m: ops.mlstm_scan(proj, 0, H * d, 2 * H * d, w, w + H, b, b, 9.0, d ** -0.5, *st, *y, cu, slots, H, d, dv, max_q=m)
        outs, constant = [(n, H, dv), (n, H)], None
    if what == "constant" and constant is None or what not in (*place, "constant"):
        pytest.skip("this recurrence has none")

    def both():
        got = []
        for m in (n, 0):
            y, st = [torch.zeros(o, device=DEV) for o in outs], [s.clone() for s in states]
            call([t.view(n, -1) for t in y], st, m)
            got.append((y, st))
        return got
    clean = both()[0][0]
    if what == "constant":
        constant[1] = odd
    else:
        t, column = place[what]
        t[at, column] = odd
    (y, st), (walk_y, walk_st) = both()
    if kind == "mlstm":                                              # its output is y / den
        clean, y, walk_y = ([o[0] / o[1][..., None]] for o in (clean, y, walk_y))
        st, walk_st = st[:2], walk_st[:2]
    for a, b in [*zip(y, walk_y), *zip(st, walk_st)]:
        assert bool((a.isfinite() == b.isfinite()).all())
        # two float recurrences of sums of up to 131 tokens, keys of 36: 1e-4 of the largest value is far above their rounding
        keep = b.isfinite()
        assert float((a - b)[keep].abs().max()) <= 1e-4 * max(1.0, float(b[keep].abs().max()))
    if what != "constant":
        for a, b in zip(y, clean):
            assert float((a[:at] - b[:at]).abs().max()) <= 1e-5 * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("scale", [1e19, 1e25])
def test_keys_whose_squares_overflow(scale):
    """A key or query whose square overflows counts as zero in both forms of the delta rule."""
    from cpmcu_amd import ops
    n, H, dk, dv = 70, 2, 36, 20
    g = torch.Generator(device=DEV).manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    qkv, gates, A, b, state = rnd(n, 2 * H * dk + H * dv), rnd(n, 2 * H), rnd(H), rnd(H), rnd(1, H, dv, dk)
    qkv[[3, 4, 66], H * dk:2 * H * dk] *= scale
    qkv[[9, 67], :H * dk] *= scale
    got = []
    for m in (n, 0):
        y, st = torch.full((n, H * dv), float("nan"), device=DEV), state.clone()
        ops.delta_scan(qkv, gates, 0, H, b, A, st, y, i32([0, n]), i32([0]), H, H, dk, dv, dk ** -0.5, max_q=m)
        got.append((y, st))
    for a, w in zip(*got):
        assert bool(w.isfinite().all()) and float((a - w).abs().max()) <= 1e-5 * float(w.abs().max())


@pytest.mark.parametrize("lens,chunks", [([33, 32, 40, 37, 64], True), ([33, 32, 40, 37, 64], False), ([1] * 8, False)])
def test_mlstm_of_more_workgroups_than_run_at_a_time(lens, chunks):
    """A carried state whose maxima differ from slot to slot and from those behind the step: every workgroup of a launch, the
    last ones too, starts from the maximum before the step.  (680 workgroups of which 256 run at a time, a walk's 2,600 and
    4,160 of which 1,024 do.)"""
    from cpmcu_amd import ops
    H, d, dv, cap = 8, 256, 512, 15.0
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    B, n, cu = len(lens), sum(lens), [0]
    for q in lens:
        cu.append(cu[-1] + q)
    slots = [(3 * i + 1) % (B + 2) for i in range(B)]
    st, ns, ms = 0.3 * rnd(B + 2, H, dv, d), 0.3 * rnd(B + 2, H, d), 4.0 * rnd(B + 2, H)
    keep, ko, vo, io, fo = [t.clone() for t in (st, ns, ms)], H * d, 2 * H * d, 2 * H * d + H * dv, 2 * H * d + H * dv + H
    proj, ib, fb = rnd(n, fo + H), rnd(H), rnd(H)
    proj[:, io:] *= 4.0
    Q, K = (proj[:, o:o + H * d].double().view(n, H, d) for o in (0, ko))
    V = proj[:, vo:vo + H * dv].double().view(n, H, dv)
    a = cap * torch.tanh((proj[:, io:io + H].double() + ib.double()) / cap)
    b = torch.nn.functional.logsigmoid(cap * torch.tanh((proj[:, fo:fo + H].double() + fb.double()) / cap))
    S, N, M = (t[slots].double() for t in (st, ns, ms))
    want, low, mag = (torch.empty(n, H, *w, dtype=torch.float64, device=DEV) for w in ((dv,), (), ()))
    for s in range(B):
        for t in range(cu[s], cu[s + 1]):
            new = torch.maximum(b[t] + M[s], a[t])
            left, take = torch.exp(b[t] + M[s] - new)[:, None], torch.exp(a[t] - new)[:, None] * K[t]
            S[s], N[s], M[s] = left[..., None] * S[s] + V[t][:, :, None] * take[:, None], left * N[s] + take, new
            qt = Q[t] * d ** -0.5
            want[t], low[t] = (S[s] * qt[:, None]).sum(-1), torch.maximum((N[s] * qt).sum(-1).abs(), torch.exp(-new)) + 1e-6
            mag[t] = (N[s] * qt).abs().sum(-1) + torch.exp(-new)
    y, den = torch.full((n, H * dv), float("nan"), device=DEV), torch.full((n, H), float("nan"), device=DEV)
    args = (proj, 0, ko, vo, io, fo, ib, fb, cap, d ** -0.5, st, ns, ms, y, den, i32(cu), i32(slots), H, d, dv)
    ops.mlstm_scan(*args, write_state=False, max_q=max(lens) if chunks else 0)
    assert all(torch.equal(x, k) for x, k in zip((st, ns, ms), keep))
    ops.mlstm_scan(*args, max_q=max(lens) if chunks else 0)
    # sums of a few hundred float products and exponentials of float sums: a few 1e-6 (y and den carry the scale of a float
    # maximum, which a walk sums up token by token); with another step's maximum a scale is off by the exponential of a
    # difference of about 4
    assert float((ms[slots].double() - M).abs().max()) <= 2e-5
    scale_out = torch.exp(ms[slots].double() - M)
    errs = [float((x - w).norm() / w.norm()) for x, w in ((st[slots].double() * scale_out[..., None, None], S),
                                                          (ns[slots].double() * scale_out[..., None], N))]
    assert max(errs) <= 1e-5, errs
    off = (y.view(n, H, dv).double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert float(off.max()) <= 1e-4 and bool(((den.double() - low).abs() <= 1e-4 * mag).all()), (float(off.max()), errs)
    others = [i for i in range(B + 2) if i not in slots]
    assert all(torch.equal(x[others], k[others]) for x, k in zip((st, ns, ms), keep))
