"""CPU: which batches the planner deals to the workgroups by length (256 compute units are assumed)."""
import pytest


@pytest.mark.parametrize("heads,kv,d,lens,balanced", [
    (32, 8, 128, [400] * 8, 0), (32, 8, 128, [800] * 8, 1), (32, 8, 128, [4000] * 24, 1), (32, 8, 128, [800] * 24, 0),
    (32, 8, 128, [30000] * 64, 0), (8, 1, 128, [400] * 2, 0), (8, 1, 128, [800] * 2, 1), (8, 1, 128, [800] * 24, 0),
    (8, 1, 128, [1600] * 24, 1), (28, 4, 128, [100] * 4, 0), (16, 4, 256, [100] * 8, 0), (16, 4, 256, [400] * 8, 1),
    (32, 8, 64, [400] * 8, 0), (32, 8, 64, [800] * 8, 1), (32, 8, 128, [8192] * 16, 1), (32, 32, 128, [8192] * 4, 0)])
def test_short_sequences_are_not_balanced(heads, kv, d, lens, balanced):
    """The plan (host arithmetic) for the longest of these lengths; the figures beside balancing_pays."""
    from tidaldecode_amd._lib import DecodePlan, lib

    plan = DecodePlan(0, 0, 0, 0, -1, -1, 0, 0)
    assert lib.td_decode_make_plan(len(lens), heads, kv, d, 1, max(lens), plan) == 0
    assert plan.balanced == balanced and plan.max_splits <= 64
