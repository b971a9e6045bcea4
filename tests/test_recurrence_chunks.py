"""Which sequences of a step a recurrence takes in chunks (CPU)."""
import random

import pytest

from cpmcu_amd import ops


@pytest.mark.parametrize("kind,workgroups", [("ssm", 256), ("delta", 128), ("mlstm", 136), ("ssm", 4)])
def test_the_chosen_are_the_longest(kind, workgroups):
    rng = random.Random(workgroups)
    for _ in range(200):
        lens = [int(2 ** rng.uniform(0, 10)) for _ in range(rng.randint(1, 80))]
        chunk_from, n = ops.recurrence_chunks(kind, lens, workgroups)
        assert n == sum(q >= chunk_from for q in lens) if n else chunk_from == 0
        if max(lens) < ops.RECURRENCES[kind].least:
            assert n == 0


def test_both_sides_of_the_rule():
    """The measured times beside the rule: one prompt alone, many equal ones, one prompt beside decoding sequences."""
    for kind, wg in (("ssm", 256), ("delta", 128), ("mlstm", 136)):
        for q in (64, 300, 2000):
            assert ops.recurrence_chunks(kind, [q], wg) == (q, 1)
        assert ops.recurrence_chunks(kind, [1] * 64, wg) == (0, 0)
        assert ops.recurrence_chunks(kind, [400] + [1] * 31, wg) == (400, 1)
    assert ops.recurrence_chunks("ssm", [64] * 32, 256) == (64, 32)
    assert ops.recurrence_chunks("ssm", [96] * 64, 256) == (0, 0)
    assert ops.recurrence_chunks("delta", [96] * 32, 128) == (0, 0)
    assert ops.recurrence_chunks("delta", [256] * 8, 128) == (256, 8)
    assert ops.recurrence_chunks("mlstm", [256] * 16, 136) == (256, 16)
