"""Buckets of recorded steps."""

from __future__ import annotations

import pytest

from mini_infer_amd.engine.decode_graph import bucket_of, mixed_bucket_of


@pytest.mark.parametrize("minimum", [1, 16])
def test_mixed_buckets_hold_their_values_and_are_seldom_a_third_too_large(minimum):
    buckets = {mixed_bucket_of(value, minimum) for value in range(1, 257)}
    assert buckets == {b for b in (1, 2, 4, 8, 16, 32, 48, 64, 96, 128, 192, 256) if b >= minimum}
    for value in range(1, 257):
        bucket = mixed_bucket_of(value, minimum)
        assert bucket == min(b for b in buckets if b >= value) <= bucket_of(value, minimum)
        assert value <= 32 or bucket < 1.5 * value
