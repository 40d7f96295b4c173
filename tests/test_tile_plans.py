"""How products of some tens to some hundreds of rows are cut into tiles: the plan is made on the host, so it is tested there."""

from __future__ import annotations

import pytest

from mini_infer_amd.ops import kernels


@pytest.mark.parametrize("cus", [256, 128, 64, 32])
def test_a_plan_counts_the_compute_units_of_its_device(cus):
    """A part of a device has fewer blocks to fill it with: sums whose order depends on the matrix alone take a block a compute unit, and
    a product is cut no finer, and expected to take longer, on fewer."""
    for n, k in ((2048, 8192), (1024, 4096), (3072, 3072)):
        _, _, ranges = kernels._tiles_plan(24, n, k, False, 16, True, 0.0, 0.0, cus)
        steps, wanted = -(-k // 64), max(1, min(16, k // 64 // 4, cus // -(-n // 64)))
        each = -(-steps // wanted)
        assert ranges == -(-steps // each)
    whole = kernels._tiles_plan(64, 4096, 4096, False, 16, False, 0.0, 0.0, 256)
    part = kernels._tiles_plan(64, 4096, 4096, False, 16, False, 0.0, 0.0, cus)
    assert part[0] >= whole[0] and part[2] <= whole[2] and (cus == 256) == (part == whole)
    assert kernels._tiles_plan(64, 4096, 4096, False, 16, False, 0.0, 0.0) == whole
