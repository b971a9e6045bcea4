"""How many columns a workgroup of the kernel for wide values takes: the rule against the workgroups it makes, one by one."""
import random

import pytest

from cpmcu_amd import ops


@pytest.fixture(autouse=True)
def mi355x(monkeypatch):
    monkeypatch.setattr(ops, "_cu_count", 256)


def share(q_lens, kv_lens, per, chunk, window, keep_first):
    """(workgroups, keys that all read over keys that 256 CUs would read if each read the longest one's)."""
    read = []
    for n, end in zip(q_lens, kv_lens):
        for a in range(end - n, end, per):
            own = [min(p % chunk + 1 if chunk else p + 1, window + keep_first if window else 1 << 30) for p in range(a, min(a + per, end))]
            read.append((sum(own) / len(own), max(own)))
    return len(read), sum(r for r, _ in read) / (256 * max(m for _, m in read))


def test_a_few_tokens_behind_a_long_history_decide():
    rule = lambda q, kv, **mask: ops.attention_wide_columns(q, 32, 1, 576, 512, kv, **mask)
    assert rule([], []) == 64 and rule([200] * 8 + [0], [200] * 9) == 128               # (a sequence without tokens brings nothing)
    assert rule([200] * 8, [200] * 8) == 128 and rule([200] * 8, [200] * 7 + [3000]) == 64
    q = [49, 202, 173, 266, 422, 26, 45, 230]
    assert rule(q, [n + h for n, h in zip(q, [2423, 2617, 0, 0, 0, 544, 1205, 0])]) == 64       # 173 us, with 128 columns 214
    assert rule([2048], [2048]) == rule([2048], [4096]) == 128 and rule([1000], [1000]) == 64
    assert rule([1280, 4], [1280, 9000]) == 64 and rule([1280, 4], [1280, 9000], window=1024) == 128
    assert rule([1280, 4], [1280, 8000], chunk=2048) == 64 and rule([1280, 4], [1280, 8000], chunk=256) == 128


def test_the_rule_counts_what_the_workgroups_read():
    rng = random.Random(3)
    seen = set()
    for _ in range(400):
        nh, q = rng.choice([8, 16, 32, 64]), [rng.randint(1, 900) for _ in range(rng.randint(1, 8))]
        kv = [n + rng.choice([0, 0, rng.randint(0, 3000)]) for n in q]
        mask = rng.choice([{}, {"chunk": rng.randint(1, 2500)}, {"window": rng.randint(1, 2500), "keep_first": rng.choice([0, 0, 100])}])
        workgroups, part = share(q, kv, 128 // nh, mask.get("chunk", 0), mask.get("window", 0), mask.get("keep_first", 0))
        got = ops.attention_wide_columns(q, nh, 1, 576, 512, kv, **mask)
        seen.add(got)
        # (a sequence's last workgroup, of fewer tokens, counts as its average one)
        if workgroups < 320 or part < 0.57:
            assert got == 64, (nh, q, kv, mask, workgroups, part)
        elif part > 0.63:
            assert got == 128, (nh, q, kv, mask, workgroups, part)
    assert seen == {64, 128}
