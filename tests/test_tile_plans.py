"""How products of some tens to some hundreds of rows are cut into tiles: the plan is made on the host, so it is tested there."""

from __future__ import annotations

import math

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


@pytest.mark.parametrize("m", [17, 24, 32, 48, 64, 100, 128, 129, 200])
@pytest.mark.parametrize("n", [2048, 4096, 8192, 10240])
@pytest.mark.parametrize("k", [4096, 8192, 14336, 16384])
@pytest.mark.parametrize("partial_ok", [False, True])
def test_few_rows_are_not_cut_into_ranges_that_begin_4_kb_apart_in_rows_of_16(m, n, k, partial_ok):
    """All blocks would ask the same memory channels; more rows, and rows of W of other lengths, are cut as before."""
    _, _, ranges = kernels._tiles_plan(m, n, k, False, 16, False, 0.0 if partial_ok else 4.0, m * n * 4 / 5e6)
    apart = -(-(k // 64) // ranges) * 128  # bytes
    assert ranges == 1 or m > 128 or k % 8192 or apart % 8192 != 4096
    if (m, n, k) == (17, 8192, 8192):
        assert ranges == 2
    if (m, n, k) == (200, 4096, 8192):
        assert ranges == 4


@pytest.mark.parametrize("n,k", [(5120, 3072), (6144, 4096), (6144, 3072), (5120, 5120), (3072, 8192)])
def test_whole_tiles_of_large_matrices_end_at_288_rows(n, k):
    """Where the library was measured faster; cut ones and small matrices go on to 320."""
    assert kernels.tiles_for(288, n, k, False) is not None
    for m in (289, 300, 320):
        plan = kernels.tiles_for(m, n, k, False)
        assert plan is None or plan[1] > 1
    assert kernels.tiles_for(320, 3072, 3072, False) is not None and kernels.tiles_for(320, 2048, 8192, True)[1] > 1


def test_gated_products_of_more_than_160_rows_take_no_tiles_above_192_by_128():
    """Larger ones were measured slower than the library from there on."""
    for n, k in ((14336, 4096), (28672, 8192), (8192, 3072), (8192, 2048), (2048, 3072)):
        assert kernels.gated_tiles_for(160, n, k) is not None
        for m in (161, 176, 192, 193, 200, 256):
            shape = kernels.gated_tiles_for(m, n, k)
            assert shape is None or math.prod(kernels.tile_size(shape)) <= 192 * 128
    assert kernels.gated_tiles_for(193, 14336, 4096) is None and kernels.gated_tiles_for(192, 14336, 4096) is not None


@pytest.mark.parametrize("counts, weight_rows, k, cuts", [
    ([4] * 16, 4096, 3072, [(0, 1, 4, 64)] * 16),
    ([100] * 16, 3072, 2048, [(0, 1, 100, 128)] * 16),
    ([150, 40] * 8, 4096, 3072, [(0, 1, 150, 160), (0, 1, 40, 64)] * 8),         # each expert the smallest form that holds its pairs
    ([250] * 16, 4096, 3072, [(0, 1, 250, 256)] * 16),
    ([0, 0, 1, 0], 256, 64, [(0, 0, 0, 64)] * 2 + [(0, 1, 1, 64), (0, 0, 0, 64)]),
    ([0, 0], 256, 64, [(0, 0, 0, 64)] * 2),                                      # nobody chose any: nothing to do
    ([1, 300, 45], 512, 512, [(0, 1, 1, 64), (0, 3, 100, 128), (0, 1, 45, 64)]),  # few tiles: smaller ones
    ([10000], 28672, 4096, [(39, 1, 16, 64)]),                                   # many: full ones and the smallest for the rest
])
def test_expert_tiles_by_what_their_launch_takes(counts, weight_rows, k, cuts):
    assert kernels.expert_tile_cuts(counts, weight_rows, k) == cuts


@pytest.mark.parametrize("counts", [[1], [63, 64, 65], [255, 256, 257, 0, 1025], [160, 161, 320, 321, 512, 513], [7] * 200, [5000, 1, 0, 2049]])
@pytest.mark.parametrize("weight_rows, k, cus", [(64, 64, 8), (4096, 3072, 256), (28672, 4096, 256), (640, 512, 64)])
def test_expert_tiles_hold_every_pair(counts, weight_rows, k, cus):
    for pairs, (full, tiles, each, rows) in zip(counts, kernels.expert_tile_cuts(counts, weight_rows, k, cus)):
        assert rows in (64, 128, 160, 256) and each <= rows
        assert full * 256 + tiles * each >= pairs > full * 256 or pairs == full == tiles == 0



@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("m, n, k", [(2048, 14336, 4096), (1777, 14336, 4096), (2048, 28672, 4096), (321, 64, 64), (4096, 4096, 14336), (700, 5000, 192),
                                     (3000, 12288, 3072), (1, 1, 64), (100000, 128, 64)])
def test_tiles_that_take_turns_cover_a_product_once(m, n, k, gated):
    """What the launch works out block by block, over its plan: every row tile of every feature tile, whole or in as many parts as it is cut into."""
    (rows, features, rest, whole, places), micros = kernels.turns_plan(m, n, k, gated)
    row_tiles, feature_tiles = -(-m // rows), -(-n // (features // 2 if gated else features))
    cut = rows // rest
    assert rows % rest == 0 and micros > 0 and places == -(-row_tiles * feature_tiles // 8) and whole % 32 == 0 and places - whole < 32
    seen = {}
    for block in range(8 * (whole + (places - whole) * cut)):
        xcd, at = block % 8, block // 8
        part = at >= whole
        place = xcd * places + (whole + (at - whole) // cut if part else at)
        if place >= min((xcd + 1) * places, row_tiles * feature_tiles):
            continue
        band = place // (8 * feature_tiles)
        in_band = min(8, row_tiles - band * 8)
        left = place - band * 8 * feature_tiles
        r0 = (band * 8 + left % in_band) * rows + ((at - whole) % cut * rest if part else 0)
        seen.setdefault((r0, left // in_band), []).append(rest if part else rows)
    made = {}
    for (r0, tile), sizes in seen.items():
        assert len(sizes) == 1 and 0 <= tile < feature_tiles
        for r in range(r0, r0 + sizes[0], 64 if sizes[0] % 64 == 0 else 32):
            assert (r, tile) not in made
            made[(r, tile)] = True
    step = 64 if rows % 64 == 0 and rest % 64 == 0 else 32
    assert len(made) == row_tiles * rows // step * feature_tiles


def test_the_rest_of_a_product_is_cut_where_whole_tiles_leave_units_idle():
    assert kernels.turns_plan(2048, 14336, 4096, gated=True)[0] == [256, 256, 128, 96, 112]
    assert kernels.turns_plan(1777, 14336, 4096, gated=True)[0] == [256, 256, 64, 96, 98]
    assert kernels.turns_plan(4096, 14336, 4096, gated=True)[0][2:] == [256, 224, 224]


@pytest.mark.parametrize("m, n, k, taken", [(321, 3072, 3072, False), (401, 3072, 3072, True), (320, 28672, 4096, False), (640, 4096, 14336, False),
                                            (2048, 4096, 14336, True), (1501, 2048, 8192, False), (2048, 2048, 8192, True), (512, 4096, 4128, False)])
def test_products_that_go_to_the_tiles_that_take_turns(m, n, k, taken):
    assert kernels.turns_pay(m, n, k) == taken


@pytest.mark.parametrize("m, n, k, kept", [(2048, 8192, 8192, True), (2049, 8192, 8192, False), (2048, 8193, 64, False), (321, 32768, 64, True), (321, 32769, 64, False),
                                           (400, 4096, 8256, False), (1501, 5120, 3072, True), (1501, 16384, 3072, False), (65536, 256, 64, True)])
def test_products_whose_order_of_sums_is_the_libraries_too(m, n, k, kept):
    """Whole tiles of 256 x 256 are counted, and against the units that the device has."""
    assert kernels.turns_keep_the_order(m, n, k) == kept
    assert not kernels.turns_keep_the_order(m, n, k, 1) or m * n <= 256 * 256


@pytest.mark.parametrize("m, n, k, gated, plain", [
    (512, 2048, 2048, True, False), (900, 2048, 2048, True, True), (768, 4096, 4096, True, False), (900, 4096, 4096, True, True), (1501, 1024, 3072, True, False),
    (512, 4097, 3072, True, True), (512, 3072, 3136, True, True), (512, 3072, 1472, True, True), (500, 512, 512, True, True), (2048, 4096, 14336, True, True),
    (640, 4096, 14336, False, False)])
def test_plain_products_with_few_outputs_for_their_k_are_the_librarys(m, n, k, gated, plain):
    """With an activation or a rotation, whose launch is saved, they stay in tiles."""
    assert kernels.turns_pay(m, n, k) == gated and kernels.plain_turns_pay(m, n, k) == plain


@pytest.mark.parametrize("m, n, k, made", [
    (271, 5120, 3072, "whole"), (100, 6144, 4096, "whole"), (100, 10240, 8192, None),       # as `linear` has them: whole tiles, K cut
    (33, 2304, 768, "own"), (320, 3072, 2048, "own"), (300, 15360, 5120, "own"), (100, 768, 3072, "own"), (100, 1536, 4096, "own"),
    (100, 512, 4096, None), (64, 768, 8192, None), (320, 512, 14336, None),                 # a block would walk a long K alone
    (33, 768, 3072, None), (64, 1536, 4096, None), (64, 2048, 3072, "own"), (65, 768, 3072, "own"),  # `linear` in ranges, or eight waves
    (300, 16384, 4096, None), (321, 2304, 768, None), (400, 768, 3072, None)])
def test_tiles_of_rotary_products(m, n, k, made):
    plan = kernels.tiles_for(m, n, k, False)
    shape = kernels.rotary_tiles_for(m, n, k)
    assert (shape is None) == (made is None)
    if made == "whole":
        assert plan == (shape, 1)
    elif made == "own":
        assert plan is None and kernels.tile_size(shape)[0] > 0


@pytest.mark.parametrize("m, n, k, linear", [(64, 3072, 3072, "cut"), (96, 4096, 4096, "cut"), (48, 4096, 2048, "rows"), (64, 3072, 2048, "rows"), (80, 3072, 2048, "whole"),
                                             (100, 3072, 3072, "whole"), (200, 3072, 2048, "whole")])
def test_rotary_products_whose_plain_ones_are_made_otherwise(m, n, k, linear):
    """Whole tiles, whatever `linear` by itself takes, which with the rotation's launch behind it is slower."""
    small = kernels.small_product_plan(m, n, k)
    form, shape, ranges = (None, *kernels.tiles_for(m, n, k, False)) if small is None else small
    assert linear == ("rows" if form is not None else "whole" if ranges == 1 else "cut")
    rotary = kernels.rotary_tiles_for(m, n, k)
    assert rotary is not None and (linear != "whole" or rotary == shape)


@pytest.mark.parametrize("m, n, k, plan", [
    (16, 2048, 2048, None), (17, 2048, 2048, "rows"), (32, 1024, 1024, "rows"), (128, 2048, 2048, "rows"), (64, 3072, 2048, "rows"),
    (192, 3072, 2048, "whole"), (320, 1024, 1024, "whole"), (321, 1024, 1024, None),                                   # small matrices
    (64, 2048, 3072, "cut"), (96, 2048, 3072, None), (64, 3072, 3072, "cut"), (97, 4096, 4096, None),                  # a longer K
    (17, 8192, 4096, "rows"), (32, 8192, 3072, "rows"), (33, 8192, 3072, None), (32, 28672, 4096, None)])             # more features
def test_products_with_small_matrices(m, n, k, plan):
    check_small_plan(m, n, k, plan)


@pytest.mark.parametrize("m, n, k, lines, plan", [
    (29, 497, 8192, True, None), (29, 496, 8192, True, "cut"), (35, 1434, 3072, True, None), (45, 2046, 2048, True, "rows"), (80, 3070, 2560, True, "whole"),
    (200, 3071, 2048, True, "whole"), (64, 2730, 4096, True, None),                              # features that no range writes four at a time
    (20, 512, 1024, False, None), (40, 512, 2000, False, None), (40, 512, 480, False, "whole"), (40, 1024, 1024, False, "whole"), (24, 2050, 1024, False, None),
    (40, 2050, 1024, False, "whole"), (24, 2048, 1024, False, "whole"), (64, 3072, 3072, False, "cut"), (24, 8192, 3072, False, None)])  # rows of W off whole lines
def test_products_with_small_matrices_that_are_not_multiples(m, n, k, lines, plan):
    check_small_plan(m, n, k, plan, lines)


def check_small_plan(m, n, k, plan, lines=True):
    got = kernels.small_product_plan(m, n, k, lines=lines)
    made = None if got is None else "rows" if got[0] is not None else "whole" if got[2] == 1 else "cut"
    assert made == plan


@pytest.mark.parametrize("tokens, experts, top, width, ff, gated, pays", [
    (1, 16, 2, 2048, 2048, True, False), (400, 16, 2, 2048, 2048, True, False), (2048, 16, 2, 2048, 2048, True, False), (4096, 64, 6, 2048, 1024, True, False),
    (400, 4, 2, 1024, 4096, True, False), (1000, 4, 2, 1024, 4096, True, True), (4096, 4, 2, 1024, 4096, True, True), (4096, 8, 2, 2048, 4096, True, True),
    (3, 64, 1, 512, 256, False, False), (4096, 4, 4, 512, 4096, False, True)])
def test_float32_experts_of_many_rows_are_sorted(monkeypatch, tokens, experts, top, width, ff, gated, pays):
    """On both sides of the line (measured at its rule), through the layer's own choice where a step is not recorded."""
    import torch

    from mini_infer_amd import ops
    from mini_infer_amd.parts import feed_forward

    assert kernels.sorted_f32_experts_pay(tokens * top, experts, width, ff, gated) == pays
    layer = feed_forward.RoutedExperts(width, ff, experts, top, torch.float32, "cpu", activation="silu_gated" if gated else "squared_relu")
    rows = 2 * ff if gated else ff
    layer.gate_up, layer.down = torch.empty((experts, rows, width), device="meta"), torch.empty((experts, width, ff), device="meta")
    x = torch.empty((tokens, width), device="meta")

    class Step:
        host_cu_seqlens_q = [0, tokens]

    for name, answer in {"expert_tiles_take": False, "expert_lines_take_f32": True, "experts_by_expert_take": True}.items():
        monkeypatch.setattr(ops, name, lambda *a, answer=answer: answer)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert layer._grouped(x, Step) == pays


@pytest.mark.parametrize("pairs, experts, k, features, gated, fours", [
    (1, 16, 2048, 2048, True, False), (12, 64, 2048, 2048, True, True), (24, 16, 2048, 2048, True, True), (47, 16, 2048, 2048, True, True), (48, 16, 2048, 2048, True, False),
    (12, 64, 512, 8192, True, False), (2, 16, 2048, 512, False, True), (2, 16, 2048, 512, True, False), (2, 16, 1024, 512, False, False), (1, 1, 4096, 4096, False, True)])
def test_which_float32_experts_are_read_for_four_rows(pairs, experts, k, features, gated, fours):
    assert kernels.f32_experts_by_fours(pairs, experts, k, features, gated) == fours


@pytest.mark.parametrize("kind, dim, heads, vdim, requests, tokens, longest, walked, chunked", [
    ("delta", 96, 31, 256, 59, 208, 115, 325, 155), ("per_channel", 200, 22, 512, 18, 302, 265, 408, 188), ("delta", 64, 14, 256, 39, 328, 218, 123, 57),
    ("per_head", 128, 15, 256, 29, 532, 191, 108, 60), ("per_head", 128, 48, 64, 1, 2048, 2048, 730, 113), ("delta", 128, 32, 128, 32, 95, 64, 110, 60),
    ("per_head", 128, 48, 64, 16, 256, 16, 32, 36), ("delta", 128, 32, 128, 100, 400, 4, 264, 399), ("delta", 128, 32, 128, 16, 128, 8, 65, 82)])
def test_scans_go_the_way_that_was_measured_to_be_faster(kind, dim, heads, vdim, requests, tokens, longest, walked, chunked):
    """Single tokens beside one portion and beside several, of which only the longest is known, prompts, and short portions (microseconds as measured)."""
    expected = kernels.scan_times(kind, tokens, requests, longest, heads, dim, vdim)
    assert kernels.chunked_scan_pays(*expected, heads * vdim) == (chunked < walked)
