"""Each HIP kernel alone against a plain reference, at other sizes than the engine's tiny models."""

import math

import numpy as np
import pytest
import torch

import plain_llama as pl

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def _tol(dtype, scale=1.0):
    return (2e-5 if dtype == torch.float32 else 2e-2) * scale


def _rand(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def _off_the_cache_lines(w):
    """A contiguous copy of `w` that begins 16 bytes past a 128-byte boundary.  The weight-streaming
    products read whole cache lines where the rows of the matrix begin on such boundaries (and K
    gives every wave an even number of 32-element steps), half lines otherwise: both ways add
    the same products in the same order, so their results are equal bit for bit."""
    flat = torch.empty(w.numel() + 64, dtype=w.dtype, device=w.device)
    shift = (-(flat.data_ptr() // w.element_size()) % 64 + 8) % 64
    out = flat[shift : shift + w.numel()].view(w.shape)
    assert out.data_ptr() % 128 == 16 and out.is_contiguous()
    out.copy_(w)
    return out


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden,vocab", [(4096, 1000), (100, 301), (90, 17)])
def test_embed_gather(dtype, hidden, vocab):
    from mini_infer_amd import ops

    table = _rand(vocab, hidden, dtype=dtype)
    ids = torch.tensor([0, vocab - 1, 5, 5, vocab // 2], dtype=torch.int32, device=DEV)
    out = ops.embed_gather(table, ids)
    assert out.dtype == torch.float32
    assert torch.equal(out, table.float()[ids.long()])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [4096, 100, 90, 9000, 1000])
@pytest.mark.parametrize("tokens", [7, 300])  # few rows; the rows of a prompt's portion
def test_add_rmsnorm(dtype, hidden, tokens):
    from mini_infer_amd import ops

    eps = 3e-6
    residual = _rand(tokens, hidden, seed=1, scale=2.0)
    delta = _rand(tokens, hidden, dtype=dtype, seed=2)
    weight = (_rand(hidden, seed=3) * 0.2 + 1.0).to(dtype)
    expected_sum = residual.double() + delta.double()
    expected = pl.rms_norm(expected_sum.cpu().numpy(), weight.double().cpu().numpy(), eps)

    res = residual.clone()
    out = ops.add_rmsnorm(delta, res, weight, eps)
    assert torch.allclose(res, expected_sum.float(), atol=1e-6)  # the sum is stored, in float32
    assert np.abs(out.float().cpu().numpy() - expected).max() < _tol(dtype, 4)

    # first layer: nothing to add, residual untouched
    res = residual.clone()
    out = ops.add_rmsnorm(None, res, weight, eps)
    assert torch.equal(res, residual)
    plain = pl.rms_norm(residual.double().cpu().numpy(), weight.double().cpu().numpy(), eps)
    assert np.abs(out.float().cpu().numpy() - plain).max() < _tol(dtype, 4)

    # chosen rows only: the residual stays as it was
    rows = torch.tensor([5, 0, 5], dtype=torch.int32, device=DEV)
    res = residual.clone()
    out = ops.add_rmsnorm(delta, res, weight, eps, rows)
    assert torch.equal(res, residual) and out.shape == (3, hidden)
    assert np.abs(out.float().cpu().numpy() - expected[[5, 0, 5]]).max() < _tol(dtype, 4)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inter", [14336, 130, 7, 136])
@pytest.mark.parametrize("tokens", [5, 300])  # few rows; the rows of a prompt's portion
def test_silu_mul(dtype, inter, tokens):
    from mini_infer_amd import ops

    gate_up = _rand(tokens, 2 * inter, dtype=dtype, seed=4, scale=3.0)
    gate_up[0, 0] = 0.0
    gate_up[0, 1 % inter] = 80.0
    gate_up[1, 0] = -80.0
    out = ops.silu_mul(gate_up).float().cpu().numpy()
    g = gate_up[:, :inter].double().cpu().numpy()
    u = gate_up[:, inter:].double().cpu().numpy()
    expected = pl.silu(g) * u
    assert np.isfinite(out).all()
    assert np.abs(out - expected).max() < _tol(dtype, max(1.0, np.abs(expected).max()))
    assert out[0, 0] == 0.0


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (7, 130, 90), (65, 301, 259), (300, 96, 4096), (33, 1, 5)])
def test_gemm_f32_is_true_float32(m, n, k):
    from mini_infer_amd import ops

    a, w = _rand(m, k, seed=5), _rand(n, k, seed=6)
    out = ops.gemm_f32(a, w)
    expected = a.double() @ w.double().T
    # float32 rounding of a K-long sum; a reduced-precision matrix mode (10-bit or
    # 7-bit mantissas) would miss this bound by a factor of ten or more
    assert (out.double() - expected).abs().max() < 6e-8 * math.sqrt(k) * float(expected.abs().max()) * 4
    # a row's result does not depend on the other rows in the batch
    alone = ops.gemm_f32(a[m // 2 : m // 2 + 1].contiguous(), w)
    assert torch.equal(alone[0], out[m // 2])
    # strided rows
    wide = _rand(m, k + 3, seed=7)
    assert torch.equal(ops.gemm_f32(wide[:, :k], w), ops.gemm_f32(wide[:, :k].contiguous(), w))


@pytest.mark.parametrize("m", [1, 3, 4, 5, 8])
@pytest.mark.parametrize("n,k", [(5, 32), (8, 288), (17, 544), (2041, 1056), (2048, 4352), (2050, 2080), (2064, 4096), (9000, 256)])
def test_few_rows_of_gemm_f32_in_groups_of_four(m, n, k):
    """One and two groups of four rows, 8 and 16 features a block with a rest, runs of K of none, one, some and more slices than a stage
    holds: the bits that a row gets among 20 (which are made otherwise), and the exact product rounded once."""
    from mini_infer_amd import ops

    a, w = _rand(20, k, seed=33), _rand(n, k, seed=34)
    out, exact = ops.gemm_f32(a[:m], w), a[:m].double() @ w.double().T
    assert torch.equal(out, ops.gemm_f32(a, w)[:m])
    assert ((out.double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 1e-12 * math.sqrt(k)).all()


@pytest.mark.parametrize("m", [1, 4, 5, 8])
@pytest.mark.parametrize("n,k", [(1, 32), (8, 288), (13, 2080), (700, 4096), (64, 4352)])
def test_gated_product_of_a_few_float32_rows(m, n, k):
    """The launch with the activation in its last step (4 rows and 8, a rest of features; above 16 slices a run 8 rows go the other way)
    gives the bits of the product and `silu_mul` in turn."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import library

    x, w = _rand(m, k, seed=35), _rand(2 * n, k, seed=36, scale=k ** -0.5)
    taken = library.load().mi_gemm_f32_swiglu_takes(x.data_ptr(), k, w.data_ptr(), k, m, n, k)
    assert taken == (m <= 4 or k <= 4096)
    assert torch.equal(ops.linear_swiglu(x, w), ops.silu_mul(ops.gemm_f32(x, w)))


@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (16, 8200, 96), (17, 33, 544), (32, 100, 2048), (33, 8, 352), (64, 50, 257), (65, 130, 4096),
                                   (50, 8192, 160), (700, 6200, 100), (90, 70, 36), (80, 70, 900)])
def test_gemm_f32_kernels_and_alignments_agree(m, n, k):
    """Every kernel (few rows in 1, 2 or 4 tiles, large and small blocks) and both ways of loading (16 bytes, single values) sum
    an output in the same order: the same bits, and the exact product rounded once (half an ulp, plus what 64-bit sums lose)."""
    from mini_infer_amd import ops

    a, w = _rand(m, k, seed=31), _rand(n, k, seed=32)
    out = ops.gemm_f32(a, w)
    exact = a.double() @ w.double().T
    assert ((out.double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 1e-12 * math.sqrt(k)).all()
    for rows in (1, 16, 17, 40, 65):
        if rows < m:
            assert torch.equal(ops.gemm_f32(a[:rows], w), out[:rows]), rows
    odd_a, odd_w = torch.zeros(m, k + 1, device=DEV), torch.zeros(n, k + 3, device=DEV)
    odd_a[:, 1:], odd_w[:, 3:] = a, w
    assert torch.equal(ops.gemm_f32(odd_a[:, 1:], odd_w[:, 3:]), out)


@pytest.mark.parametrize(
    "m,n,k",
    [(1, 4096, 4096), (8, 6144, 4096), (16, 96, 64), (7, 301, 96), (13, 130, 160), (16, 1000, 14336),
     (5, 128256, 256), (3, 7, 32), (9, 28672, 4096), (2, 16400, 1056), (4, 4096, 1536), (6, 640, 3072), (16, 2050, 512)],
)
def test_gemm_skinny_bf16(m, n, k):
    from mini_infer_amd import ops

    a, w = _rand(m, k, dtype=torch.bfloat16, seed=9), _rand(n, k, dtype=torch.bfloat16, seed=10, scale=0.05)
    out = ops.gemm_skinny_bf16(a, w)
    expected = a.double() @ w.double().T
    # float32 accumulation of exact bfloat16 products, one rounding to bfloat16 at the end
    assert (out.double() - expected).abs().max() < 2.0 ** -8 * float(expected.abs().max()) + 1e-6
    # a row's result does not depend on the other rows in the batch
    alone = ops.gemm_skinny_bf16(a[m // 2 : m // 2 + 1].contiguous(), w)
    assert torch.equal(alone[0], out[m // 2])
    # strided activations (a slice of a wider buffer), and the dispatch in `linear`
    wide = _rand(m, k + 8, dtype=torch.bfloat16, seed=11)
    assert torch.equal(ops.gemm_skinny_bf16(wide[:, :k], w), ops.gemm_skinny_bf16(wide[:, :k].contiguous(), w))
    assert torch.equal(ops.linear(a, w), out)
    assert torch.equal(ops.gemm_skinny_bf16(a, _off_the_cache_lines(w)), out)


@pytest.mark.parametrize(
    "m,n,k",
    [(1, 4096, 14336), (8, 1000, 8192 + 32), (16, 4096, 4096), (17, 1003, 4096), (33, 136, 608), (64, 4096, 14336),
     (47, 5, 32), (64, 260, 8192 - 224), (128, 4096, 4096), (101, 200, 1024 + 64), (24, 3072, 8192 + 64)],
)
def test_linear_in_partial_sums_then_norm_is_linear_then_norm(m, n, k):
    """A product left as sums over ranges of K, added up by the norm that follows it: the
    same residual and output, bit for bit, as with the pieces added first (`finish`), and the
    product itself within float32 accumulation of the exact one; a row's pieces do not
    depend on the other rows."""
    from mini_infer_amd import ops

    a, w = _rand(m, k, dtype=torch.bfloat16, seed=31), _rand(n, k, dtype=torch.bfloat16, seed=32, scale=0.05)
    partial = ops.linear_partial_sums(a, w)
    assert partial.pieces.dtype == torch.float32 and partial.pieces.shape[1:] == (m, n)
    delta = partial.finish()
    expected = a.double() @ w.double().T
    assert (delta.double() - expected).abs().max() < 2.0 ** -8 * float(expected.abs().max()) + 1e-6
    alone = ops.linear_partial_sums(a[m // 2 : m // 2 + 1].contiguous(), w)
    assert torch.equal(alone.pieces[:, 0], partial.pieces[:, m // 2])
    # strided activations: a slice of a wider buffer
    wide = _rand(m, k + 8, dtype=torch.bfloat16, seed=35)
    assert torch.equal(ops.linear_partial_sums(wide[:, :k], w).pieces, ops.linear_partial_sums(wide[:, :k].contiguous(), w).pieces)
    assert torch.equal(ops.linear_partial_sums(a, _off_the_cache_lines(w)).pieces, partial.pieces)
    weight = _rand(n, dtype=torch.bfloat16, seed=33).abs() + 0.5
    for rows in (None, torch.tensor([m - 1, 0], dtype=torch.int32, device=DEV)):
        res_a, res_b = _rand(m, n, seed=34), _rand(m, n, seed=34)
        out_a = ops.add_rmsnorm(partial, res_a, weight, 1e-5, rows)
        out_b = ops.add_rmsnorm(delta, res_b, weight, 1e-5, rows)
        assert torch.equal(out_a, out_b) and torch.equal(res_a, res_b)


TILE_SHAPES = 14


def test_every_tile_shape_is_tested():
    from mini_infer_amd.ops import kernels

    sizes = [kernels.tile_size(shape) for shape in range(TILE_SHAPES + 1)]
    assert len(set(sizes)) == TILE_SHAPES + 1 and sizes[-1] == (0, 0)


@pytest.mark.parametrize("shape", range(TILE_SHAPES))
def test_products_in_tiles(shape):
    """Every shape at the edges of its tiles, whole, over ranges of K, as float32 times a number, and gated with each activation; K of one step, of fewer steps than
    the ring has stages, of odd 32s, and of ranges of unequal length; rows of a wider buffer, whose values beside and behind the result
    stay, on boundaries of four values and off them; a row of infinities stays alone."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    bm, bn = kernels.tile_size(shape)
    cases = [(bm, bn, 64, 1), (bm + 1, bn + 1, 128, 2), (bm - 1, bn - 3, 320, 1), (2 * bm + 5, 2 * bn + 4, 64 * 11, 3), (1, 5, 32, 1),
             (17, bn + 62, 96, 1), (bm, 70, 64 * 7 + 32, 2), (3, 2 * bn, 1024, 16)]

    def made(kind, a, w, n, dtype, ranges=1, scale=1.0, spare=0, bias=None):
        """The product in the first columns of rows with `spare` more (over ranges: [ranges, m, n], contiguous) before more values."""
        m = a.shape[0]
        if kind == 1:
            flat = torch.full((ranges * m * n + 64,), 7.0, device=DEV)
            out, rest = flat[:-64].view(ranges, m, n), [flat[-64:]]
        else:
            wide = torch.full((m + 1, n + spare), 7.0, dtype=dtype, device=DEV)
            out, rest = wide[:m, :n], [wide[:, n:], wide[m:]]
        kernels._tiles(kind, a, w, out, n, shape, ranges, scale, bias, 2.5, 1.702)
        assert all((each == 7).all() for each in rest), (kind, a.shape, n, ranges, spare)
        return out

    for m, n, k, ranges in cases:
        a = _rand(m, k + 8, dtype=torch.bfloat16, seed=41)[:, :k]
        w = _rand(2 * n, k, dtype=torch.bfloat16, seed=42, scale=0.05)
        if m > 2:
            a[m - 1] = float("inf")
        finite = slice(0, m - 1 if m > 2 else m)
        exact = (a.double() @ w.double().T)[finite]
        # (exact products in float32 sums of k terms and the ranges', each rounded or cut; then one rounding to 8 bits)
        summed = 2.0 ** -23 * (k + ranges) * (a.double().abs() @ w.double().abs().T)[finite] + 1e-30
        rounded = summed + 2.0 ** -8 * exact.abs()
        pieces = made(1, a, w, 2 * n, torch.float32, ranges)
        assert ((pieces.double().sum(0)[finite] - exact).abs() <= summed).all(), (m, n, k)
        if ranges == 1:
            outs = [made(0, a, w, 2 * n, torch.bfloat16, spare=spare) for spare in (0, 3, -2 * n % 4 + 4)]
            out = outs[0]
            assert all(torch.equal(other[finite], out[finite]) for other in outs)
            assert ((out[finite].double() - exact).abs() <= rounded).all(), (m, n, k)
            for spare in (0, 1, -2 * n % 4):
                assert torch.equal(made(2, a, w, 2 * n, torch.float32, scale=0.25, spare=spare)[finite], out.float()[finite] * 0.25)
            g, u = out.double()[finite, :n], out.double()[finite, n:]
            wanted = g / (1.0 + torch.exp(-g)) * u
            for spare in (0, 3, -n % 4 + 4):
                # (a product may come out one rounding apart: the gated tile sums the same pieces in the same order, so it does not)
                gated = made(3, a, w, n, torch.bfloat16, spare=spare)[finite]
                assert ((gated.double() - wanted).abs() <= 2.0 ** -8 * wanted.abs() + 1e-30).all(), (m, n, k)
                # (and the other activations are those of the launch that would follow)
                bias = _rand(2 * n, seed=48)
                assert torch.equal(made(4, a, w, n, torch.bfloat16, spare=spare, bias=bias)[finite], ops.clamped_glu(out, bias, 2.5, 1.702)[finite])
                assert torch.equal(made(4, a, w, n, torch.bfloat16, spare=spare)[finite], ops.clamped_glu(out, None, 2.5, 1.702)[finite])
                assert torch.equal(made(5, a, w, n, torch.bfloat16, spare=spare)[finite], ops.gated_mul(out[:, :n], out[:, n:], "gelu_tanh")[finite])


@pytest.mark.parametrize("shape", [0, 1, 3, 6, 9, 11, 13])
@pytest.mark.parametrize("k", [64, 192, 480, 2048])
def test_tiles_that_begin_a_step_later_than_their_neighbours(shape, k):
    """An output head and gated products whose rows of W are 4 KB apart: more tiles than steps of K, K of one step and, which begins like the others, of odd 32s."""
    from mini_infer_amd.ops import kernels

    bm, bn = kernels.tile_size(shape)
    check_tiles_of_rows_4_kb_apart(shape, bm + 3, bn * (35 if bn <= 64 else 5), k)


@pytest.mark.parametrize("shape", range(14))
@pytest.mark.parametrize("k, row_tiles, feature_tiles", [(2048, 1, 129), (2048, 2, 131), (256, 1, 200), (64, 1, 210), (4096, 1, 130)])
def test_many_tiles_that_begin_a_step_later_than_their_neighbours(shape, k, row_tiles, feature_tiles):
    """On the side of the rule where they do (some of these, by the width and the rows of their tiles, begin like the others)."""
    from mini_infer_amd.ops import kernels

    bm, bn = kernels.tile_size(shape)
    check_tiles_of_rows_4_kb_apart(shape, bm * row_tiles - 1, bn // 2 * feature_tiles - 3, k, stride=max(k, 2048))


def check_tiles_of_rows_4_kb_apart(shape, m, n, k, stride=2048):
    from mini_infer_amd.ops import kernels

    a, w = _rand(m, k, dtype=torch.bfloat16, seed=71), _rand(2 * n, stride, dtype=torch.bfloat16, seed=72, scale=0.05)[:, :k]
    exact = a.double() @ w.double().T
    # (as test_products_in_tiles: sums of k terms, one rounding to 8 bits; in the activation half a unit of each factor and of the result)
    summed = 2.0 ** -23 * (k + 1) * (a.double().abs() @ w.double().abs().T) + 1e-30
    logits = kernels._tiles(2, a, w, torch.empty(m, 2 * n, device=DEV), 2 * n, shape, 1, 0.25)
    assert ((logits.double() * 4 - exact).abs() <= summed + 2.0 ** -8 * exact.abs()).all()
    gated = kernels._tiles(3, a, w, torch.empty(m, n, dtype=torch.bfloat16, device=DEV), n, shape, 1).double()
    g, u = exact[:, :n], exact[:, n:]
    off_g, off_u = (e + 2.0 ** -8 * x.abs() for e, x in ((summed[:, :n], g), (summed[:, n:], u)))
    wanted = torch.nn.functional.silu(g) * u  # (|silu'| <= 1.1, |silu(g)| <= |g|)
    assert ((gated - wanted).abs() <= 1.1 * off_g * (u.abs() + off_u) + g.abs() * off_u + 2.0 ** -8 * wanted.abs() + 1e-6).all()


def test_every_form_of_the_tiles_that_take_turns_is_tested():
    from mini_infer_amd.ops import library

    lib = library.load()
    assert lib.mi_gemm_turns_rows(10) > 0 and lib.mi_gemm_turns_rows(11) == 0


@pytest.mark.parametrize("form", range(-1, 11))
def test_products_in_tiles_that_take_turns(form):
    """Every form (-1: the plan's) at the edges of its tiles, plain and with each activation; K of one step, of fewer steps than the ring has stages and of
    more; rows of a wider buffer, whose values beside and behind the result stay, on boundaries of eight values and off them; more row tiles
    than stand side by side; a row of infinities stays alone."""
    from mini_infer_amd import ops
    from mini_infer_amd.exceptions import KernelShapeError
    from mini_infer_amd.ops import kernels, library

    lib = library.load()
    bm, bn = (lib.mi_gemm_turns_rows(form), lib.mi_gemm_turns_features(form)) if form >= 0 else (256, 256)
    half = bn // 2
    cases = [(bm, half, 64), (bm + 1, half + 1, 128), (bm - 1, half - 3, 192), (2 * bm + 5, bn + 4, 320), (1, 5, 64), (9 * bm + 3, 70, 64 * 9)]
    if form < 0:
        cases += [(512, 16896, 64), (1000, 14400, 64)]  # (both cut the tiles of the last round)
        assert any(kernels.turns_plan(m, 2 * n, k)[0][0] != kernels.turns_plan(m, 2 * n, k)[0][2] for m, n, k in cases)

    def made(act, a, w, n, spare=0, bias=None):
        m = a.shape[0]
        wide = torch.full((m + 1, n + spare), 7.0, dtype=torch.bfloat16, device=DEV)
        kernels._turns(act, a, w, n, bias, 3.0, 1.702, form, wide[:m, :n])
        assert (wide[:m, n:] == 7).all() and (wide[m:] == 7).all(), (act, a.shape, n, spare)
        return wide[:m, :n]

    for m, n, k in cases:
        a = _rand(m, k + 8, dtype=torch.bfloat16, seed=43)[:, :k]
        w = _rand(2 * n, k, dtype=torch.bfloat16, seed=44, scale=0.05)
        if m > 2:
            a[m - 1] = float("inf")
        finite = slice(0, m - 1 if m > 2 else m)
        exact = (a.double() @ w.double().T)[finite]
        # (float32 sums of k products, then one rounding to 8 bits)
        bound = 2.0 ** -23 * k * (a.double().abs() @ w.double().abs().T)[finite] + 2.0 ** -8 * exact.abs() + 1e-30
        out = made(kernels.TURNS_NONE, a, w, 2 * n)[finite]
        assert ((out.double() - exact).abs() <= bound).all(), (m, n, k)
        for spare in (3, -2 * n % 8 + 8):
            assert torch.equal(made(kernels.TURNS_NONE, a, w, 2 * n, spare)[finite], out)
        if form >= 0 and not lib.mi_gemm_turns_gated(form):
            with pytest.raises(KernelShapeError):
                made(kernels.TURNS_SILU, a, w, n)
            continue
        # the activation is that of the launch that would follow the product
        bias = _rand(2 * n, seed=45)
        for spare in (0, 3, -n % 8 + 8):
            assert torch.equal(made(kernels.TURNS_SILU, a, w, n, spare)[finite], ops.silu_mul(out))
            assert torch.equal(made(kernels.TURNS_GELU, a, w, n, spare)[finite], ops.gated_mul(out[:, :n], out[:, n:], "gelu_tanh"))
            assert torch.equal(made(kernels.TURNS_CLAMPED, a, w, n, spare, bias)[finite], ops.clamped_glu(out, bias, 3.0, 1.702))
            assert torch.equal(made(kernels.TURNS_CLAMPED, a, w, n, spare)[finite], ops.clamped_glu(out, None, 3.0, 1.702))


@pytest.mark.parametrize("m, n, k", [(401, 2304, 2048), (640, 1000, 512), (2048, 1500, 1024)])
def test_products_of_many_rows_go_through_the_tiles_that_take_turns(m, n, k, monkeypatch):
    """Plain and gated, from the public entry points; K that is not whole 64s, rows off 16 bytes and few rows do not."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    taken = []
    own = kernels._turns
    monkeypatch.setattr(kernels, "_turns", lambda act, *rest, **more: (taken.append(act), own(act, *rest, **more))[1])
    a, w = _rand(m, k + 40, dtype=torch.bfloat16, seed=46), _rand(2 * n, k + 40, dtype=torch.bfloat16, seed=47, scale=0.05)
    exact = a[:, :k].double() @ w[:, :k].double().T
    for steady in (False, True):
        got = ops.linear(a[:, :k], w[:, :k], steady=steady)
        assert (got.double() - exact).abs().max() < 2.0 ** -7 * exact.abs().max()
    assert taken == [kernels.TURNS_NONE] * 2
    g, u = exact[:, :n].float().bfloat16().double(), exact[:, n:].float().bfloat16().double()
    for got, want in ((ops.linear_swiglu(a[:, :k], w[:, :k]), torch.nn.functional.silu(g) * u),
                      (ops.linear_geglu(a[:, :k], w[:, :k]), torch.nn.functional.gelu(g, approximate="tanh") * u),
                      (ops.linear_clamped_glu(a[:, :k], w[:, :k], None, 2.0, 1.702), g.clamp(max=2.0) * torch.sigmoid(1.702 * g.clamp(max=2.0)) * (u.clamp(-2.0, 2.0) + 1))):
        assert (got.double() - want).abs().max() < 2.0 ** -6 * want.abs().max()
    assert taken[2:] == [kernels.TURNS_SILU, kernels.TURNS_GELU, kernels.TURNS_CLAMPED]
    del taken[:]
    ops.linear(a[:, :k - 32], w[:, :k - 32])
    ops.linear(a[:, 1:k + 1], w[:, 1:k + 1])
    ops.linear(a[:320, :k], w[:, :k])
    assert taken == []


@pytest.mark.parametrize("m, n, k", [(321, 1536, 64), (700, 520, 192), (1030, 2304, 512), (2048, 1024, 2048), (513, 4096, 576)])
def test_tiles_that_take_turns_give_the_same_bits_in_every_form(m, n, k):
    """All forms, the plan's launch, and the vendor library where it does not cut K."""
    from mini_infer_amd.ops import kernels, library

    a, w = _rand(m, k, dtype=torch.bfloat16, seed=50), _rand(n, k, dtype=torch.bfloat16, seed=51, scale=0.05)
    planned = kernels._turns(kernels.TURNS_NONE, a, w, n)
    for form in range(11):
        assert library.load().mi_gemm_turns_rows(form) > 0
        assert torch.equal(kernels._turns(kernels.TURNS_NONE, a, w, n, only=form), planned), form
    assert kernels.turns_keep_the_order(m, n, k) and torch.equal(a @ w.t(), planned)


@pytest.mark.parametrize("n, k", [(2048, 2048), (3072, 3072), (5120, 3072), (4096, 3072), (2112, 3072), (3072, 8192), (6144, 4096), (7168, 4096), (4096, 4096),
                                  (4608, 1536), (4096, 512), (16384, 3072), (28672, 4096), (4096, 14336)])
def test_steady_products_of_many_rows_are_the_librarys_bit_for_bit(n, k):
    """The matrices of routed designs, at row counts within the bounds of `turns_keep_the_order` and beyond: the library cuts K of 16384 x 3072 at 2,060
    rows, of 28672 x 4096 at 1,750, of 4096 x 14336 at 1,600."""
    from mini_infer_amd import ops

    w = _rand(n, k, dtype=torch.bfloat16, seed=53, scale=0.05)
    for m in (321, 777, 1501, 1600, 1750, 2048, 2060):
        a = _rand(m, k, dtype=torch.bfloat16, seed=52)
        want = a @ w.t()
        assert torch.equal(ops.linear(a, w, steady=True), want), m
        if m in (321, 1600, 1750):
            assert torch.equal(ops.linear_swiglu(a, w, steady=True), ops.silu_mul(want)), m


@pytest.mark.parametrize("m, n, k", [(17, 40, 64), (31, 2048, 2048), (32, 1000, 576), (33, 515, 1088), (64, 3072, 2048), (100, 258, 4160), (256, 1024, 192)])
def test_products_of_some_tens_of_rows_whose_waves_share_k(m, n, k):
    """Every form, waves without a share of K and uneven ones, strided operands, tails of rows and features; nothing is written beside the output.
    `linear` takes the planned one, and other kernels where W does not lie in whole cache lines."""
    from mini_infer_amd import ops
    from mini_infer_amd.exceptions import KernelShapeError
    from mini_infer_amd.ops import kernels, library

    lib = library.load()
    a, w = _rand(m, k + 24, dtype=torch.bfloat16, seed=61)[:, :k], _rand(n, k + 64, dtype=torch.bfloat16, seed=62, scale=0.05)[:, :k]
    exact = a.double() @ w.double().T
    # half a bfloat16 unit, and k float32 roundings of the sums of magnitudes (eight of those more where the waves meet)
    bound = exact.abs() * 2.0 ** -8 + (k + 8) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)

    def made(form, spare):
        out = torch.full((m, n + spare), 7.0, dtype=torch.bfloat16, device="cuda")
        library.check(lib.mi_gemm_rows_bf16(form, a.data_ptr(), a.stride(0), w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0), m, n, k,
                                            torch.cuda.current_stream().cuda_stream))
        assert (out[:, n:] == 7.0).all()
        return out[:, :n]

    form, first = 0, made(0, 0)
    while lib.mi_gemm_rows_rows(form):
        for spare in (0, 3, -n % 8 + 8):
            got = made(form, spare)
            assert torch.equal(got, first) and ((got.double() - exact).abs() <= bound).all(), (form, spare)
        form += 1
    assert form == 3
    with pytest.raises(KernelShapeError):
        made(form, 0)
    plan = kernels.small_product_plan(m, n, k)
    got = ops.linear(a, w)
    assert ((got.double() - exact).abs() <= bound).all()
    assert plan is None or plan[0] is None or torch.equal(got, first)
    off = _rand(n * (k + 8) + 8, dtype=torch.bfloat16, seed=63)[8:].view(n, k + 8)[:, :k].copy_(w)  # rows on 16 bytes
    assert not kernels._whole_lines(a, off) and ((ops.linear(a, off).double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("m,n,k", [(17, 3072, 3072), (33, 2048, 8192), (271, 3072, 8192), (100, 8192, 2048), (24, 1000, 8224), (400, 2048, 8192)])
def test_linear_of_some_tens_to_some_hundreds_of_rows(m, n, k):
    """`linear` through tiles, with and without a consumer for the pieces; operands that the tiles do not take (rows off 16 bytes) go on
    being taken."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    a, w = _rand(m, k, dtype=torch.bfloat16, seed=43), _rand(n, k, dtype=torch.bfloat16, seed=44, scale=0.05)
    expected = a.double() @ w.double().T
    bound = 2.0 ** -8 * float(expected.abs().max()) + 1e-6
    assert kernels.tiles_for(m, n, k, True) is not None
    left = ops.linear(a, w, partial_ok=True)
    left = left.finish() if isinstance(left, ops.PartialSums) else left
    off = _rand(m * k + 4, dtype=torch.bfloat16, seed=45)[4:].view(m, k).copy_(a)
    for got in (left, ops.linear(a, w), ops.linear(off, w)):
        assert got.dtype == torch.bfloat16 and (got.double() - expected).abs().max() < bound
    assert torch.equal(kernels.sum_pieces(_rand(3, 5, 7, seed=46)), _rand(3, 5, 7, seed=46).sum(0).bfloat16())


@pytest.mark.parametrize("count,rows,columns,first", [(1, 1, 1, 0), (2, 17, 3072, 0), (16, 70, 1030, 0), (5, 3, 7, 0), (3, 5, 7, 1), (4, 6, 8, 2)])
def test_partial_sums_finish_in_one_launch(monkeypatch, count, rows, columns, first):
    """The sum in order, rounded once, by one launch of this library; pieces off 16 bytes and columns of wider pieces by torch, the same."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import library

    lib, launches = library.load(), []
    launch = lib.mi_sum_pieces
    monkeypatch.setattr(lib, "mi_sum_pieces", lambda *a: (launches.append(a), launch(*a))[1])
    pieces = _rand(first + count, rows, columns, seed=5)[first:]
    expected = pieces[0].clone()
    for piece in pieces[1:]:
        expected += piece
    finished = ops.PartialSums(pieces, torch.bfloat16).finish()
    assert finished.dtype == torch.bfloat16 and torch.equal(finished, expected.bfloat16())
    assert len(launches) == (first * rows * columns % 4 == 0)
    wide = torch.cat([pieces, pieces], dim=2)[:, :, :columns]
    assert torch.equal(ops.PartialSums(wide, torch.bfloat16).finish(), expected.bfloat16())
    assert ops.PartialSums(pieces, torch.float32).finish().equal(expected)


def test_linear_leaves_partial_sums_only_where_asked_and_where_it_pays():
    from mini_infer_amd import ops
    from mini_infer_amd.exceptions import KernelShapeError

    a, w = _rand(12, 12288, dtype=torch.bfloat16, seed=36), _rand(64, 12288, dtype=torch.bfloat16, seed=37, scale=0.05)
    assert ops.partial_sums_pay(12, 64, 12288) and isinstance(ops.linear(a, w, partial_ok=True), ops.PartialSums)
    assert isinstance(ops.linear(a, w), torch.Tensor)
    assert not ops.partial_sums_pay(8, 64, 12288) and not ops.partial_sums_pay(12, 8192, 12288) and ops.partial_sums_pay(15, 8192, 12288)
    assert not ops.partial_sums_pay(16, 64, 4096) and ops.partial_sums_pay(17, 64, 4096)
    assert not ops.partial_sums_pay(4, 64, 12288) and not ops.partial_sums_pay(16, 3072, 8192)
    assert not ops.partial_sums_pay(129, 64, 12288) and not ops.partial_sums_pay(8, 28672, 12288)
    assert isinstance(ops.linear(a[:, :4096].contiguous(), w[:, :4096].contiguous(), partial_ok=True), torch.Tensor)
    assert isinstance(ops.linear(a.float(), w.float(), partial_ok=True), torch.Tensor)
    partial = ops.linear(a, w, partial_ok=True)
    with pytest.raises(KernelShapeError, match="partial sums"):
        ops.add_rmsnorm(ops.PartialSums(partial.pieces[:, :1].contiguous(), torch.bfloat16), _rand(8, 64),
                        _rand(64, dtype=torch.bfloat16), 1e-5)
    with pytest.raises(KernelShapeError, match="1 to 128 rows"):
        ops.linear_partial_sums(_rand(129, 64, dtype=torch.bfloat16), _rand(16, 64, dtype=torch.bfloat16))


@pytest.mark.parametrize("m, n, k", [(17, 5000, 1024), (32, 8192, 3072), (31, 5127, 2048), (18, 8193, 1536), (25, 11003, 4096), (32, 9000, 2560), (20, 8200, 5120)])
def test_gated_products_of_17_to_32_rows_in_eighths_of_k_give_the_streaming_bits(monkeypatch, m, n, k):
    """Tiles of both widths, with a last one of few features, begun at any pair of eighths or not, each row as in a product of at most 16."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    taken = []
    own = kernels._tiles
    monkeypatch.setattr(kernels, "_tiles", lambda kind, *rest, **more: (taken.append((kind, rest[5])), own(kind, *rest, **more))[1])
    a, w = _rand(m, k + 64, dtype=torch.bfloat16, seed=61)[:, :k], _rand(2 * n, k, dtype=torch.bfloat16, seed=62, scale=0.05)
    bias = _rand(2 * n, seed=63, dtype=torch.float32)
    got = [f(steady) for steady in (False, True) for f in (
        lambda s: ops.linear_swiglu(a, w, steady=s), lambda s: ops.linear_geglu(a, w, steady=s), lambda s: ops.linear_clamped_glu(a, w, bias, 2.0, 1.702, steady=s))]
    assert taken == [(3, kernels.GATED_EIGHTHS), (5, kernels.GATED_EIGHTHS), (4, kernels.GATED_EIGHTHS)] * 2
    both = torch.cat([ops.gemm_skinny_bf16(a[at:at + 16], w) for at in range(0, m, 16)])
    want = [ops.silu_mul(both), ops.gated_mul(both[:, :n], both[:, n:], "gelu_tanh"), ops.clamped_glu(both, bias, 2.0, 1.702)]
    for i, x in enumerate(got):
        assert torch.equal(x, want[i % 3]), i


@pytest.mark.parametrize(
    "m,inter,k",
    [(1, 14336, 4096), (8, 14336, 4096), (16, 160, 64), (7, 301, 96), (13, 4100, 160), (3, 5, 32), (9, 8192, 3072),
     (5, 520, 1536), (2, 24, 512), (17, 14336, 4096), (32, 8192, 3072), (24, 160, 64), (31, 301, 96), (20, 520, 1536)],
)
def test_linear_swiglu_is_the_product_followed_by_the_activation(m, inter, k):
    from mini_infer_amd import ops

    a = _rand(m, k, dtype=torch.bfloat16, seed=12)
    w = _rand(2 * inter, k, dtype=torch.bfloat16, seed=13, scale=0.08)
    fused = ops.linear_swiglu(a, w)
    assert fused.shape == (m, inter)
    # the two-kernel path: the product (rounded to bfloat16), then the activation (the plain
    # weight-streaming product takes 16 rows; a row's result does not depend on the others)
    for first in range(0, m, 16):
        assert torch.equal(fused[first : first + 16], ops.silu_mul(ops.gemm_skinny_bf16(a[first : first + 16], w)))
    assert torch.equal(ops.linear_swiglu(a, _off_the_cache_lines(w)), fused)
    gate_up = (a.double() @ w.double().T).bfloat16().double()
    gate, up = gate_up[:, :inter], gate_up[:, inter:]
    expected = gate / (1 + torch.exp(-gate)) * up
    assert (fused.double() - expected).abs().max() < 2.0 ** -7 * float(expected.abs().max()) + 1e-6
    # more rows than the fused kernel takes: the same function, through the library product
    many = _rand(40, k, dtype=torch.bfloat16, seed=14)
    assert ops.linear_swiglu(many, w).shape == (40, inter)
    # float32 goes through the true float32 product
    got32 = ops.linear_swiglu(a.float(), w.float())
    exact = a.double() @ w.double().T
    exact = exact[:, :inter] / (1 + torch.exp(-exact[:, :inter])) * exact[:, inter:]
    assert (got32.double() - exact).abs().max() < 1e-4 * float(exact.abs().max()) + 1e-6


@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize(
    "m,hidden,q_heads,kv_heads,head_dim,page_size",
    [(8, 4096, 32, 8, 128, 16), (1, 4096, 32, 8, 128, 16), (16, 96, 3, 1, 32, 16), (5, 160, 6, 2, 64, 32), (9, 64, 4, 4, 96, 48),
     (3, 1536, 6, 2, 64, 16), (17, 4096, 32, 8, 128, 16), (32, 1536, 6, 2, 64, 16), (25, 96, 3, 1, 32, 16)],
)
def test_qkv_rope_write_is_the_product_followed_by_rotation_and_cache_write(
    v_transposed, m, hidden, q_heads, kv_heads, head_dim, page_size
):
    from mini_infer_amd import ops

    num_pages = 7
    width = (q_heads + 2 * kv_heads) * head_dim
    x = _rand(m, hidden, dtype=torch.bfloat16, seed=31)
    w = _rand(width, hidden, dtype=torch.bfloat16, seed=32, scale=0.1)
    positions = torch.tensor(([0, 1, 700, 5, 131071, 17, 18, 19, 3000, 2, 4, 6, 8, 10, 12, 14] + list(range(50, 66)))[:m],
                             dtype=torch.int32, device=DEV)
    inv_freq = torch.from_numpy(pl.inv_freq_default(head_dim, 500000.0)).to(DEV)
    cos, sin = ops.rope_table(positions, inv_freq)
    slots = torch.tensor(([40, 3, 17, 16, 0, 43, -1, 9, 22, 5, 6, 7, 30, 31, 32, 33] + list(range(60, 76)))[:m],
                         dtype=torch.int32, device=DEV)
    slots = torch.where(slots >= 0, slots % (num_pages * page_size), slots)
    assert len(set(slots[slots >= 0].tolist())) == int((slots >= 0).sum())  # (no two rows write one slot)

    def pages():
        k = torch.full((num_pages, kv_heads, page_size, head_dim), 7.0, dtype=torch.bfloat16, device=DEV)
        v_shape = (num_pages, kv_heads, head_dim, page_size) if v_transposed else k.shape
        return k, torch.full(v_shape, 7.0, dtype=torch.bfloat16, device=DEV)

    k_two, v_two = pages()
    qkv = torch.cat([ops.gemm_skinny_bf16(x[first : first + 16], w) for first in range(0, m, 16)])
    ops.rope_kv_write(qkv, cos, sin, slots, k_two, v_two, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                      rotary_dim=head_dim, interleaved=False, v_transposed=v_transposed)
    k_one, v_one = pages()
    queries = ops.qkv_rope_write(x, w, cos, sin, slots, k_one, v_one, q_heads=q_heads, kv_heads=kv_heads,
                                 head_dim=head_dim, v_transposed=v_transposed)
    assert queries.shape == (m, q_heads * head_dim)
    # the same products rounded the same way, the same rotation formula: equal up to how the
    # compiler contracts a multiply-add before the final rounding
    tol = 2.0 ** -7 * float(qkv.float().abs().max())
    assert (queries.float() - qkv[:, : q_heads * head_dim].float()).abs().max() <= tol
    assert (k_one.float() - k_two.float()).abs().max() <= tol
    assert torch.equal(v_one, v_two)  # values are copied, not rotated
    k_off, v_off = pages()
    off_lines = ops.qkv_rope_write(x, _off_the_cache_lines(w), cos, sin, slots, k_off, v_off, q_heads=q_heads,
                                   kv_heads=kv_heads, head_dim=head_dim, v_transposed=v_transposed)
    assert torch.equal(off_lines, queries) and torch.equal(k_off, k_one) and torch.equal(v_off, v_one)
    # queries only (a layer that reads another layer's keys and values): pages stay untouched
    k_none, v_none = pages()
    only_q = ops.qkv_rope_write(x, w[: q_heads * head_dim], cos, sin, None, k_none, v_none, q_heads=q_heads,
                                kv_heads=0, head_dim=head_dim, v_transposed=v_transposed)
    assert torch.equal(only_q, queries)
    assert torch.all(k_none == 7.0) and torch.all(v_none == 7.0)


def test_linear_falls_back_to_the_library_where_the_skinny_kernel_does_not_apply():
    from mini_infer_amd import ops
    from mini_infer_amd.exceptions import KernelShapeError

    a, w = _rand(5, 90, dtype=torch.bfloat16), _rand(40, 90, dtype=torch.bfloat16, seed=1)
    assert (ops.linear(a, w).double() - a.double() @ w.double().T).abs().max() < 0.2
    big = _rand(100, 64, dtype=torch.bfloat16)
    assert ops.linear(big, _rand(32, 64, dtype=torch.bfloat16, seed=2)).shape == (100, 32)
    with pytest.raises(KernelShapeError, match="m <= 16"):
        ops.gemm_skinny_bf16(big, _rand(32, 64, dtype=torch.bfloat16, seed=2))
    with pytest.raises(KernelShapeError):
        ops.gemm_skinny_bf16(a, w)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(
    "q_heads,kv_heads,head_dim,rotary_dim,interleaved",
    [(32, 8, 128, 128, False), (3, 1, 32, 32, False), (6, 3, 48, 16, False), (4, 2, 64, 64, True), (2, 2, 16, 0, False),
     (5, 1, 40, 24, False)],
)
@pytest.mark.parametrize("tokens", [9, 300])  # few rows; the rows of a prompt's portion
def test_rope_kv_write(dtype, q_heads, kv_heads, head_dim, rotary_dim, interleaved, tokens):
    from mini_infer_amd import ops

    page_size = 4
    num_pages = tokens + 2
    width = (q_heads + 2 * kv_heads) * head_dim
    qkv = _rand(tokens, width, dtype=dtype, seed=8)
    original = qkv.clone()
    rng = np.random.default_rng(tokens)
    some = [0, 1, 2, 3, 700, 701, 5, 6, 131071]
    positions = torch.tensor(some + rng.integers(0, 131072, tokens - len(some)).tolist(), dtype=torch.int32, device=DEV)
    half = rotary_dim // 2
    if half:
        inv_freq = torch.from_numpy(pl.inv_freq_default(rotary_dim, 500000.0)).to(DEV)
        cos, sin = ops.rope_table(positions, inv_freq)
        angle = positions.float().cpu().numpy()[:, None] * inv_freq.cpu().numpy()[None, :]
        assert np.abs(cos.cpu().numpy() - np.cos(angle.astype(np.float64))).max() < 2e-6
        assert np.abs(sin.cpu().numpy() - np.sin(angle.astype(np.float64))).max() < 2e-6
    else:
        cos = sin = torch.empty((tokens, 0), dtype=torch.float32, device=DEV)
    # scattered slots, one token not written at all
    more = [int(x) for x in rng.permutation(num_pages * page_size) if x not in (40, 3, 17, 16, 0, 43, 9, 22)]
    slots = torch.tensor([40, 3, 17, 16, 0, 43, -1, 9, 22] + more[: tokens - 9], dtype=torch.int32, device=DEV)
    k_pages = torch.zeros((num_pages, kv_heads, page_size, head_dim), dtype=dtype, device=DEV)
    v_pages = torch.zeros_like(k_pages)
    ops.rope_kv_write(qkv, cos, sin, slots, k_pages, v_pages, q_heads=q_heads, kv_heads=kv_heads,
                      head_dim=head_dim, rotary_dim=rotary_dim, interleaved=interleaved)
    # the same write with values transposed inside each page
    vt_pages = torch.zeros((num_pages, kv_heads, head_dim, page_size), dtype=dtype, device=DEV)
    ops.rope_kv_write(original.clone(), cos, sin, slots, torch.zeros_like(k_pages), vt_pages, q_heads=q_heads,
                      kv_heads=kv_heads, head_dim=head_dim, rotary_dim=rotary_dim, interleaved=interleaved,
                      v_transposed=True)
    assert torch.equal(vt_pages.transpose(2, 3), v_pages)

    def rotate(x):  # x [T, heads, D] float64
        if not half:
            return x
        c, s = cos.double().cpu().numpy()[:, None, :], sin.double().cpu().numpy()[:, None, :]
        out = x.copy()
        if interleaved:
            x0, x1 = x[..., 0:rotary_dim:2], x[..., 1:rotary_dim:2]
            out[..., 0:rotary_dim:2], out[..., 1:rotary_dim:2] = x0 * c - x1 * s, x1 * c + x0 * s
        else:
            x0, x1 = x[..., :half], x[..., half:rotary_dim]
            out[..., :half], out[..., half:rotary_dim] = x0 * c - x1 * s, x1 * c + x0 * s
        return out

    src = original.double().cpu().numpy()
    q_in = src[:, : q_heads * head_dim].reshape(tokens, q_heads, head_dim)
    k_in = src[:, q_heads * head_dim : (q_heads + kv_heads) * head_dim].reshape(tokens, kv_heads, head_dim)
    v_in = src[:, (q_heads + kv_heads) * head_dim :].reshape(tokens, kv_heads, head_dim)
    got_q = qkv[:, : q_heads * head_dim].double().cpu().numpy().reshape(tokens, q_heads, head_dim)
    assert np.abs(got_q - rotate(q_in)).max() < _tol(dtype, 4)
    assert torch.equal(qkv[:, q_heads * head_dim :], original[:, q_heads * head_dim :])  # k, v inputs untouched
    expect_k = np.zeros(k_pages.shape)
    expect_v = np.zeros(v_pages.shape)
    rk = rotate(k_in)
    for t, slot in enumerate(slots.tolist()):
        if slot >= 0:
            expect_k[slot // page_size, :, slot % page_size] = rk[t]
            expect_v[slot // page_size, :, slot % page_size] = v_in[t]
    assert np.abs(k_pages.double().cpu().numpy() - expect_k).max() < _tol(dtype, 4)
    assert np.array_equal(v_pages.double().cpu().numpy(), expect_v)  # values copied bit for bit, other slots still zero
    if half:
        # position 0 leaves q as it was
        assert torch.equal(qkv[0, : q_heads * head_dim], original[0, : q_heads * head_dim])


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("q_heads,kv_heads,head_dim,rotary_dim,extra,writes", [
    (24, 8, 128, 128, 0, True), (3, 1, 64, 32, 4, True), (4, 2, 72, 8, 0, True), (8, 2, 64, 64, 0, False)])
@pytest.mark.parametrize("tokens,pieces", [(1, 2), (17, 3), (700, 16)])
def test_rope_kv_write_of_a_projection_in_pieces(q_heads, kv_heads, head_dim, rotary_dim, extra, writes, transposed, tokens, pieces):
    """The bits of the same with the pieces added up first (`PartialSums.finish`): whole heads and parts rotated, pages filled whole and
    not, a token without a slot, a step that writes nothing."""
    from mini_infer_amd import ops

    page, width = 16, (q_heads + 2 * kv_heads) * head_dim + extra
    sums = ops.PartialSums(_rand(pieces, tokens, width, seed=1), torch.bfloat16)
    cos, sin = _rand(tokens, rotary_dim // 2, seed=2), _rand(tokens, rotary_dim // 2, seed=3)
    slots = torch.arange(5, tokens + 5, dtype=torch.int32, device=DEV)
    slots[tokens // 2] = -1
    results = []
    for qkv in (sums, sums.finish()):
        k_pages = torch.zeros((tokens // page + 2, kv_heads, page, head_dim), dtype=torch.bfloat16, device=DEV)
        v_pages = torch.zeros_like(k_pages.transpose(2, 3).contiguous() if transposed else k_pages)
        queries = ops.rope_kv_write(qkv, cos, sin, slots if writes else None, k_pages, v_pages, q_heads=q_heads, kv_heads=kv_heads if writes else 0,
                                    head_dim=head_dim, rotary_dim=rotary_dim, v_transposed=transposed)
        results.append((queries[:, : q_heads * head_dim], k_pages, v_pages))
    assert all(torch.equal(a, b) for a, b in zip(*results)) and bool(results[0][1].any()) == (writes and tokens > 1)


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,rotary_dim", [(5, 1, 20, 16), (3, 1, 100, 40), (7, 7, 12, 8)])
def test_rope_kv_write_in_pieces_of_rows_that_are_not_whole_16_bytes(q_heads, kv_heads, head_dim, rotary_dim):
    """Queries whose heads together are an odd number of 8 bytes: taken like any others that `rope_takes_partial_sums` answers for."""
    from mini_infer_amd import ops

    tokens, page, width = 20, 16, (q_heads + 2 * kv_heads) * head_dim
    assert q_heads * head_dim % 8 == 4 and ops.rope_takes_partial_sums(head_dim, rotary_dim, False)
    sums = ops.PartialSums(_rand(3, tokens, width, seed=1), torch.bfloat16)
    cos, sin = _rand(tokens, rotary_dim // 2, seed=2), _rand(tokens, rotary_dim // 2, seed=3)
    slots = torch.arange(tokens, dtype=torch.int32, device=DEV)
    results = []
    for qkv in (sums, sums.finish()):
        k_pages = torch.zeros((2, kv_heads, page, head_dim), dtype=torch.bfloat16, device=DEV)
        v_pages = torch.zeros((2, kv_heads, head_dim, page), dtype=torch.bfloat16, device=DEV)
        queries = ops.rope_kv_write(qkv, cos, sin, slots, k_pages, v_pages, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                                    rotary_dim=rotary_dim, v_transposed=True)
        results.append((queries[:, : q_heads * head_dim], k_pages, v_pages))
    assert all(torch.equal(a, b) for a, b in zip(*results)) and results[0][1].any()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("page_size", [16, 8])
@pytest.mark.parametrize("more_pages", [0, 40])  # 40 more whole pages: the rows of a prompt's portion
def test_rope_kv_write_whole_pages_of_transposed_values(dtype, page_size, more_pages):
    """Tokens that fill a page in order have their transposed values written a whole page at a
    time by the page's first token; pages filled out of order, from the middle, or only in
    part go token by token.  All give what the plain layout gives, transposed."""
    from mini_infer_amd import ops

    q_heads, kv_heads, head_dim, num_pages = 4, 2, 32, 7 + more_pages
    ps = page_size
    slots = (
        list(range(2 * ps, 3 * ps))  # page 2, in order: written at once
        + [0 * ps + i for i in np.random.default_rng(0).permutation(ps)]  # page 0, out of order
        + list(range(4 * ps + 3, 4 * ps + 3 + 5))  # page 4 from its middle
        + list(range(5 * ps, 5 * ps + ps // 2))  # half of page 5
        + [-1]  # a token that is not written
        + list(range(6 * ps, 7 * ps))  # page 6, in order, at the very end of the step
        + list(range(3 * ps, 3 * ps + ps - 1))  # page 3 but for its last slot
        + list(range(7 * ps, (7 + more_pages) * ps))  # (a token too late to start on a page's edge)
    )
    tokens = len(slots)
    qkv = _rand(tokens, (q_heads + 2 * kv_heads) * head_dim, dtype=dtype, seed=21)
    positions = torch.arange(tokens, dtype=torch.int32, device=DEV)
    cos, sin = ops.rope_table(positions, torch.from_numpy(pl.inv_freq_default(head_dim, 10000.0)).to(DEV))
    slot_t = torch.tensor(slots, dtype=torch.int32, device=DEV)
    k_a = torch.zeros((num_pages, kv_heads, ps, head_dim), dtype=dtype, device=DEV)
    v_a = torch.zeros_like(k_a)
    ops.rope_kv_write(qkv.clone(), cos, sin, slot_t, k_a, v_a, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                      rotary_dim=head_dim, interleaved=False)
    k_b = torch.zeros_like(k_a)
    v_b = torch.zeros((num_pages, kv_heads, head_dim, ps), dtype=dtype, device=DEV)
    ops.rope_kv_write(qkv.clone(), cos, sin, slot_t, k_b, v_b, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                      rotary_dim=head_dim, interleaved=False, v_transposed=True)
    assert torch.equal(k_a, k_b) and torch.equal(v_b.transpose(2, 3), v_a)
    values = qkv[:, (q_heads + kv_heads) * head_dim :].reshape(tokens, kv_heads, head_dim)
    for t, slot in enumerate(slots):
        if slot >= 0:
            assert torch.equal(v_a[slot // ps, :, slot % ps], values[t])
    assert int((v_a != 0).any(dim=-1).sum()) == sum(1 for s in slots if s >= 0) * kv_heads  # nothing else was written


def _paged_case(dtype, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=0, v_transposed=False):
    """Random keys/values scattered over shuffled pages; queries are the last q_len positions."""
    rng = np.random.default_rng(seed)
    num_requests = len(lengths)
    pages_per = [-(-n // page_size) for n in lengths]
    num_pages = sum(pages_per) + 3
    order = rng.permutation(num_pages)
    max_blocks = max(pages_per)
    table = np.full((num_requests, max_blocks), -1, dtype=np.int32)
    k_pages = torch.zeros((num_pages, kv_heads, page_size, head_dim), dtype=dtype)
    v_pages = torch.zeros_like(k_pages)
    ks, vs, qs, token_request, positions = [], [], [], [], []
    at = 0
    for b, n in enumerate(lengths):
        table[b, : pages_per[b]] = order[at : at + pages_per[b]]
        at += pages_per[b]
        k = torch.from_numpy(rng.standard_normal((n, kv_heads, head_dim))).to(dtype)
        v = torch.from_numpy(rng.standard_normal((n, kv_heads, head_dim))).to(dtype)
        at_page = torch.from_numpy(table[b, np.arange(n) // page_size].astype(np.int64))
        at_slot = torch.arange(n) % page_size
        k_pages[at_page, :, at_slot] = k
        v_pages[at_page, :, at_slot] = v
        q = torch.from_numpy(rng.standard_normal((q_lens[b], q_heads, head_dim))).to(dtype)
        ks.append(k), vs.append(v), qs.append(q)
        token_request += [b] * q_lens[b]
        positions += list(range(n - q_lens[b], n))
    cu = [0]
    for n in q_lens:
        cu.append(cu[-1] + n)
    if v_transposed:
        v_pages = v_pages.transpose(2, 3).contiguous()
    return dict(
        q=torch.cat(qs).reshape(-1, q_heads * head_dim).to(DEV), qs=qs, ks=ks, vs=vs,
        k_pages=k_pages.to(DEV), v_pages=v_pages.to(DEV), v_transposed=v_transposed,
        cu=torch.tensor(cu, dtype=torch.int32, device=DEV), host_cu=cu,
        block_table=torch.from_numpy(table).to(DEV),
        token_request=torch.tensor(token_request, dtype=torch.int32, device=DEV),
        positions=torch.tensor(positions, dtype=torch.int32, device=DEV),
    )


def _attend(case, q_heads, kv_heads, head_dim, scale, window, max_seq_len):
    from mini_infer_amd import ops

    return ops.paged_attention(
        case["q"], case["k_pages"], case["v_pages"], case["block_table"], case["token_request"],
        case["positions"], case["cu"], case["host_cu"], q_heads=q_heads, kv_heads=kv_heads,
        head_dim=head_dim, scale=scale, window=window, max_seq_len=max_seq_len,
        v_transposed=case["v_transposed"])


def _attention_expected(case, scale, window):
    outs = []
    for q, k, v in zip(case["qs"], case["ks"], case["vs"]):
        out = pl.causal_attention(q.double().numpy(), k.double().numpy(), v.double().numpy(), scale, window)
        outs.append(out.reshape(out.shape[0], -1))
    return np.concatenate(outs)


ATTENTION_MODES = [("plain", torch.float32), ("plain", torch.bfloat16), ("mfma", torch.bfloat16)]
PLAIN_SHAPES = [
    (32, 8, 128, 16, None),
    (5, 5, 64, 1, None),
    (7, 1, 16, 4, None),
    (6, 2, 48, 8, 9),
    (10, 2, 80, 64, None),
    (4, 4, 256, 16, 40),
    (12, 2, 112, 32, None),
    # head sizes no 16-byte load divides: read in pairs of elements, every row's end guarded
    (8, 2, 100, 16, None),
    (6, 3, 40, 4, 21),
    (3, 1, 2, 4, None),
    (4, 2, 130, 16, None),
    (5, 1, 254, 8, 50),
]
MFMA_SHAPES = [
    (32, 8, 128, 16, None),
    (3, 1, 32, 16, None),
    (7, 1, 64, 32, None),
    (6, 2, 96, 16, 9),
    (40, 2, 64, 16, None),
    (8, 2, 256, 64, 40),
    (12, 4, 192, 16, None),
    (5, 5, 128, 48, 70),
]


def _attention_cases():
    for mode, dtype in ATTENTION_MODES:
        for shape in MFMA_SHAPES if mode == "mfma" else PLAIN_SHAPES:
            yield pytest.param(mode, dtype, *shape, id=f"{mode}-{str(dtype)[6:]}-" + "-".join(map(str, shape)))


@pytest.mark.parametrize("mode,dtype,q_heads,kv_heads,head_dim,page_size,window", list(_attention_cases()))
def test_paged_attention_mixed_batch(mode, dtype, q_heads, kv_heads, head_dim, page_size, window):
    """Portions of prompts beside single tokens, pages in shuffled order, groups of 1 to 20 heads."""
    lengths, q_lens = [70, 1, 33, 129, 64, 200], [70, 1, 5, 1, 2, 37]
    case = _paged_case(dtype, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=head_dim,
                       v_transposed=mode == "mfma")
    scale = 1.0 / math.sqrt(head_dim)
    out = _attend(case, q_heads, kv_heads, head_dim, scale, window, max(lengths))
    expected = _attention_expected(case, scale, window)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(dtype, 2)


@pytest.mark.parametrize("mode,dtype", ATTENTION_MODES)
@pytest.mark.parametrize("q_heads,kv_heads,window", [(8, 2, None), (40, 2, None), (4, 4, 1000)])
def test_paged_attention_decode_only_splits_keys(mode, dtype, q_heads, kv_heads, window):
    """Single tokens over long contexts: the key range is split over blocks and recombined."""
    from mini_infer_amd import ops

    head_dim, page_size = 128, 16
    lengths, q_lens = [3000, 517, 1, 64, 2049], [1, 1, 1, 1, 1]
    assert ops.attention_splits(5 * kv_heads, max(lengths)) > 1
    case = _paged_case(dtype, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=1,
                       v_transposed=mode == "mfma")
    scale = 0.2
    out = _attend(case, q_heads, kv_heads, head_dim, scale, window, max(lengths))
    expected = _attention_expected(case, scale, window)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(dtype, 2)


@pytest.mark.parametrize("mode,dtype", ATTENTION_MODES)
def test_paged_attention_portion_over_long_context_splits_keys(mode, dtype):
    """A short portion late in a long prompt: few tiles, so keys are split there too."""
    q_heads, kv_heads, head_dim, page_size = 8, 2, 64, 16
    lengths, q_lens = [2500, 900], [40, 3]
    case = _paged_case(dtype, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=2,
                       v_transposed=mode == "mfma")
    out = _attend(case, q_heads, kv_heads, head_dim, 0.15, None, max(lengths))
    expected = _attention_expected(case, 0.15, None)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(dtype, 2)


@pytest.mark.parametrize("mode,dtype", ATTENTION_MODES)
def test_paged_attention_single_tokens_first_then_portions(mode, dtype):
    """The order a scheduler produces: decoding requests (one token each, long and short
    contexts) first, portions of prompts after them.  The matrix-core path runs the two
    runs of requests as two launches over the same buffers."""
    q_heads, kv_heads, head_dim, page_size = 8, 2, 64, 16
    lengths, q_lens = [1500, 17, 640, 300, 90, 33], [1, 1, 1, 140, 90, 2]
    case = _paged_case(dtype, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=4,
                       v_transposed=mode == "mfma")
    out = _attend(case, q_heads, kv_heads, head_dim, 0.15, None, max(lengths))
    expected = _attention_expected(case, 0.15, None)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(dtype, 2)


def test_float32_attention_over_thousands_of_keys_is_rounded_once():
    """The 32-bit path's attention keeps its sums in 64-bit: the output of a row over 2,500 keys
    differs from the exact one by about one float32 rounding (relative 2.5e-8 on average).  A
    float32 sum that is rounded at every key is 6e-7 away at this length, which 32 layers
    turn into logits off by more than 1e-4."""
    q_heads, kv_heads, head_dim, page_size = 8, 2, 128, 16
    lengths, q_lens = [2500, 1800], [300, 1]
    case = _paged_case(torch.float32, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=9)
    scale = 0.35  # scores of a few units either way: some keys stand out, hundreds still count
    out = _attend(case, q_heads, kv_heads, head_dim, scale, None, max(lengths)).double().cpu().numpy()
    expected = _attention_expected(case, scale, None)
    relative = np.linalg.norm(out - expected) / np.linalg.norm(expected)
    assert relative < 6e-8, f"relative error {relative:.2e}"


@pytest.mark.parametrize("m,n,k", [(1, 1000, 256), (8, 333, 96), (16, 4100, 512)])
def test_product_with_float32_output_keeps_its_sums(m, n, k):
    """The output head's product for few bfloat16 rows writes float32 itself: the values of
    `gemm_skinny_bf16`, widened (what the many-row path gives too)."""
    from mini_infer_amd import ops

    a, w = _rand(m, k, dtype=torch.bfloat16, seed=1).to(DEV), _rand(n, k, dtype=torch.bfloat16, seed=2).to(DEV)
    got = ops.linear_f32_out(a, w)
    assert got.dtype == torch.float32 and got.shape == (m, n)
    exact = a.double() @ w.double().T
    assert float((got.double() - exact).abs().max()) < _tol(torch.bfloat16) * k ** 0.5
    assert torch.equal(got, ops.gemm_skinny_bf16(a, w).float())
    # float32 operands and many rows go their own ways to the same kind of result
    assert ops.linear_f32_out(a.float(), w.float()).dtype == torch.float32
    many = _rand(40, k, dtype=torch.bfloat16, seed=3).to(DEV)
    assert ops.linear_f32_out(many, w).dtype == torch.float32


def test_float32_product_is_rounded_once():
    """`gemm_f32` carries its sums in 64-bit: a sum over 14,336 terms is one float32 rounding
    away from exact (2.5e-8 on average), in the many-row and in the few-row kernel alike."""
    from mini_infer_amd import ops

    a = _rand(40, 14336, seed=1).to(DEV)
    w = _rand(96, 14336, seed=2).to(DEV)
    exact = a.double() @ w.double().T
    for rows in (40, 7):
        got = ops.gemm_f32(a[:rows], w).double()
        relative = float((got - exact[:rows]).norm() / exact[:rows].norm())
        assert relative < 4e-8, f"{rows} rows: relative error {relative:.2e}"
    assert torch.equal(ops.gemm_f32(a[:7], w), ops.gemm_f32(a, w)[:7])  # a row's bits do not depend on its company


@pytest.mark.parametrize("mode,dtype", ATTENTION_MODES)
@pytest.mark.parametrize("q_heads,kv_heads,head_dim,window", [(8, 2, 64, None), (32, 8, 128, 50), (6, 3, 96, None)])
def test_paged_attention_with_request_boundaries_known_on_the_device_only(mode, dtype, q_heads, kv_heads, head_dim, window):
    """What a recorded step with portions in it asks of the attention: `host_cu_seqlens_q=None`,
    the launch shaped by the number of tokens and requests alone; requests that bring no token
    (here two, at the end, as the padding of a bucket leaves them) are passed over."""
    from mini_infer_amd import ops

    page_size = 16
    lengths, q_lens = [300, 41, 1500, 90, 64], [70, 1, 1, 33, 2]
    case = _paged_case(dtype, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=21, v_transposed=mode == "mfma")
    tokens = case["q"].shape[0]
    cu = torch.tensor(case["host_cu"] + [tokens, tokens], dtype=torch.int32, device=DEV)
    table = torch.cat([case["block_table"], torch.zeros((2, case["block_table"].shape[1]), dtype=torch.int32, device=DEV)])
    scale = 1.0 / math.sqrt(head_dim)
    out = ops.paged_attention(
        case["q"], case["k_pages"], case["v_pages"], table, case["token_request"], case["positions"], cu, None,
        q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, scale=scale, window=window, max_seq_len=2048,
        v_transposed=case["v_transposed"])
    expected = _attention_expected(case, scale, window)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(dtype, 2)


@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(8, 2, 64), (3, 3, 30), (10, 2, 128), (4, 1, 98)])
@pytest.mark.parametrize("lengths", [[1], [63, 64, 65], [255, 256, 257, 300], [1, 2, 130, 511, 1030]])
def test_paged_attention_float32_four_waves_a_range(q_heads, kv_heads, head_dim, lengths):
    """Few decoded tokens in 32 bits: four waves share a range's keys (none, one or several 64s each, the last one short) and
    are merged in 64 bits.  A weight of a key is rounded to float32 once (2^-24 relative), so is the result: 4e-7 of the largest
    value leaves those two, and the partial results of cut ranges, room to add up."""
    page_size = 16
    case = _paged_case(torch.float32, q_heads, kv_heads, head_dim, page_size, lengths, [1] * len(lengths), seed=41)
    scale = 1.0 / math.sqrt(head_dim)
    out = _attend(case, q_heads, kv_heads, head_dim, scale, None, max(lengths))
    expected = _attention_expected(case, scale, None)
    assert np.abs(out.double().cpu().numpy() - expected).max() < 4e-7 * max(1.0, np.abs(expected).max())


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,window", [(32, 8, 64, None), (24, 8, 128, None), (40, 2, 128, 130), (3, 3, 64, 40)])
@pytest.mark.parametrize("lengths,q_lens", [
    ([1, 2], [1, 2]), ([300, 33, 600], [1, 1, 256]), ([2000, 1, 31, 900, 700, 50], [1, 1, 1, 40, 200, 1]), ([90, 43, 3000], [1, 43, 85]),
])
@pytest.mark.parametrize("on_device", [False, True])
def test_paged_attention_of_portions_beside_single_tokens_in_one_launch(monkeypatch, q_heads, kv_heads, head_dim, window, lengths, q_lens, on_device):
    """Both parts whole and in key ranges, tiles of 42, 16 and 128 tokens with and without rests, a single token behind the portions (on the
    device it has a decode block, else a tile); boundaries known and found on the device, there with a request that brings nothing.
    Sinks, caps, slopes, chunks and gates: as in launches of their own, but for the ranges' order (bfloat16 results)."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, 16, lengths, q_lens, seed=17, v_transposed=True)
    lib, taken = kernels.library.load(), []
    launch = lib.mi_attn_mixed
    monkeypatch.setattr(lib, "mi_attn_mixed", lambda *a: (taken.append(a[10]), launch(*a))[1])
    tokens, scale = case["q"].shape[0], head_dim ** -0.5
    table, cu, host_cu, held = case["block_table"], case["cu"], case["host_cu"], list(lengths)
    if on_device:
        table, cu, host_cu, held = torch.cat([table, torch.zeros_like(table[:1])]), torch.cat([cu, cu[-1:]]), None, None

    def attend(**more):
        return ops.paged_attention(case["q"], case["k_pages"], case["v_pages"], table, case["token_request"], case["positions"], cu, host_cu,
                                   q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, scale=scale, window=window, max_seq_len=max(lengths),
                                   v_transposed=True, host_seq_lens=held, **more)

    leading = next(i for i, n in enumerate(q_lens) if n > 1)
    got = attend()
    assert taken == [-1 if on_device else leading]
    assert np.abs(got.double().cpu().numpy() - _attention_expected(case, scale, window)).max() < _tol(torch.bfloat16, 2)
    options = {"sinks": _rand(q_heads, seed=1), "softcap": 5.0, "slopes": _rand(q_heads, seed=2).abs() * 0.02, "chunk": 100,
               "gate": _rand(tokens, q_heads, seed=3, dtype=torch.bfloat16)}
    wide = torch.zeros((tokens, q_heads * head_dim + 8), dtype=torch.bfloat16, device=DEV)
    got = attend(out=wide[:, 4:-4], **options)
    assert len(taken) == 2 and not wide[:, :4].any() and not wide[:, -4:].any()
    monkeypatch.setattr(lib, "mi_attn_mixed_supported", lambda *a: 0)
    assert (got.float() - attend(**options).float()).abs().max() < _tol(torch.bfloat16, 2) and len(taken) == 2


@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(6, 2, 128), (8, 1, 64)])
@pytest.mark.parametrize("lengths,q_lens", [([20000, 300], [1, 300]), ([17, 9100], [1, 150]), ([12001, 8300, 8200], [1, 1, 33])])
def test_paged_attention_of_long_contexts_beside_portions(q_heads, kv_heads, head_dim, lengths, q_lens):
    """Thousands of positions on either side, and on both, cut into their most ranges."""
    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, 16, lengths, q_lens, seed=23, v_transposed=True)
    scale = head_dim ** -0.5
    out = _attend(case, q_heads, kv_heads, head_dim, scale, None, max(lengths))
    assert np.abs(out.double().cpu().numpy() - _attention_expected(case, scale, None)).max() < _tol(torch.bfloat16, 2)


@pytest.mark.parametrize("lengths,q_lens", [([30, 20], [1, 0]), ([300, 20, 900, 1], [1, 1, 0, 0]), ([30, 20, 9], [1, 0, 1]), ([600, 70, 300], [1, 0, 70])])
def test_paged_attention_of_single_tokens_before_requests_without_tokens(lengths, q_lens):
    """Boundaries known to the host, some requests of the step without tokens behind those with one."""
    case = _paged_case(torch.bfloat16, 4, 2, 64, 16, lengths, q_lens, seed=19, v_transposed=True)
    out = _attend(case, 4, 2, 64, 0.125, None, max(lengths))
    with_tokens = [i for i, n in enumerate(q_lens) if n]
    expected = _attention_expected({key: [case[key][i] for i in with_tokens] for key in ("qs", "ks", "vs")}, 0.125, None)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(torch.bfloat16, 2)


@pytest.mark.parametrize("window", [None, 700])
def test_paged_attention_whole_long_prompts_many_tiles(window):
    """Whole prompts of a few thousand tokens beside a short one: dozens of tiles per head,
    more than fit on the GPU at once, so the order in which tiles are handed out (long and
    short ones paired) and the tile-to-request search over several requests are exercised."""
    q_heads, kv_heads, head_dim, page_size = 8, 2, 64, 16
    lengths = q_lens = [2210, 37, 300]
    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=6,
                       v_transposed=True)
    out = _attend(case, q_heads, kv_heads, head_dim, 0.12, window, max(lengths))
    expected = _attention_expected(case, 0.12, window)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(torch.bfloat16, 2)


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,page_size,window", [s for s in MFMA_SHAPES if s[2] <= 128])
@pytest.mark.parametrize("lengths,q_lens", [
    ([70, 33, 129, 64, 200], [70, 5, 1, 2, 37]),
    ([900, 37, 300], [900, 37, 300]),
    ([2500, 900, 700], [40, 3, 699]),
    ([1500, 17, 640, 300], [1, 1, 140, 90]),  # single tokens first: a launch of their own in the decode shape
])
def test_paged_attention_in_blocks_of_256_rows(monkeypatch, q_heads, kv_heads, head_dim, page_size, window, lengths, q_lens):
    """The launch shape that long prompts get (8 waves, 256 rows a block), forced here on
    short ones: mixed portions, whole prompts over many tiles, portions late in a long
    context (key ranges), groups of 1 to 20 heads; and the same through the usual shape."""
    from mini_infer_amd.ops import kernels

    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, page_size, lengths, q_lens, seed=head_dim + 1,
                       v_transposed=True)
    scale = 1.0 / math.sqrt(head_dim)
    usual = _attend(case, q_heads, kv_heads, head_dim, scale, window, max(lengths))
    monkeypatch.setattr(kernels, "WIDE_PREFILL_MIN_BLOCKS", 1)
    shapes = []
    launch = kernels.library.load().mi_attn_mfma
    monkeypatch.setattr(kernels.library.load(), "mi_attn_mfma", lambda *a: (shapes.append(a[23]), launch(*a))[1])
    wide = _attend(case, q_heads, kv_heads, head_dim, scale, window, max(lengths))
    assert shapes == [kernels.ATTN_SHAPE_DECODE] * (q_lens[0] == 1) + [kernels.ATTN_SHAPE_PREFILL_WIDE]
    expected = _attention_expected(case, scale, window)
    assert np.abs(wide.double().cpu().numpy() - expected).max() < _tol(torch.bfloat16, 2)
    assert np.abs(usual.double().cpu().numpy() - expected).max() < _tol(torch.bfloat16, 2)


@pytest.mark.parametrize("rows_per_block", [128, 256])
@pytest.mark.parametrize("window", [None, 100])
def test_paged_attention_prompt_rows_find_planted_keys(monkeypatch, rows_per_block, window):
    """A whole prompt of 1,000 tokens in both prefill shapes: for chosen (query, key) pairs the
    key is made to stand out for that query, so the query's output must be that key's value.
    The pairs sit on the diagonal, at the first and last key, on both sides of the edges of the
    32-key tiles and of the 64- and 128-token row tiles, and on the window's edge; a tile that
    is skipped or masked wrongly, which random keys would hide in the tolerance, shows."""
    from mini_infer_amd.ops import kernels

    q_heads, kv_heads, head_dim, page_size, length = 2, 1, 64, 16, 1000
    scale = 1.0 / 8.0
    pairs = [(999, 0), (998, 998), (64, 64), (65, 63), (127, 96), (128, 127), (129, 129), (500, 31), (501, 32),
             (700, 255), (701, 256), (300, 201), (330, 300), (63, 2), (257, 254)]
    if window is not None:
        pairs = [(t, p) for t, p in pairs if t - p < window] + [(999, 900), (400, 301), (161, 62), (192, 93)]
    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, page_size, [length], [length], seed=31,
                       v_transposed=True)
    assert len({p for _, p in pairs}) == len(pairs) == len({t for t, _ in pairs})
    for t, p in pairs:
        key = (case["qs"][0][t, 0].float() * 6.0).to(torch.bfloat16)  # score 6 |q|^2 / 8 = 48 +- a few
        case["ks"][0][p, 0] = key
        case["k_pages"][case["block_table"][0, p // page_size].item(), 0, p % page_size] = key.to(DEV)
    if rows_per_block == 256:
        monkeypatch.setattr(kernels, "WIDE_PREFILL_MIN_BLOCKS", 1)
    shapes = []
    launch = kernels.library.load().mi_attn_mfma
    monkeypatch.setattr(kernels.library.load(), "mi_attn_mfma", lambda *a: (shapes.append(a[23]), launch(*a))[1])
    out = _attend(case, q_heads, kv_heads, head_dim, scale, window, length)
    assert shapes == [kernels.ATTN_SHAPE_PREFILL_WIDE if rows_per_block == 256 else kernels.ATTN_SHAPE_PREFILL]
    out = out.float().cpu().reshape(length, q_heads, head_dim)
    for t, p in pairs:
        assert (out[t, 0] - case["vs"][0][p, 0].float()).abs().max() < 2e-2, (t, p)
    expected = _attention_expected(case, scale, window)
    assert np.abs(out.reshape(length, -1).double().numpy() - expected).max() < _tol(torch.bfloat16, 2)


@pytest.mark.parametrize("mode,dtype", ATTENTION_MODES)
def test_paged_attention_finds_one_far_key_and_respects_edges(mode, dtype):
    """One key among a thousand is made to stand out; the output must be its value.
    Placed at a page's first and last slot, at the causal edge and at the window's edge."""
    head_dim, page_size, length = 64, 16, 1000
    transposed = mode == "mfma"

    def plant(case, spot):
        q = case["qs"][0][0, 0].float()
        page = case["block_table"][0, spot // page_size].item()
        case["k_pages"][page, 0, spot % page_size] = (q * 4.0).to(dtype).to(DEV)  # score >> all others

    for window, spots in ((None, [0, 15, 16, 31, 32, 511, 512, 999]), (100, [900, 901, 911, 912, 927, 928, 999])):
        for spot in spots:
            case = _paged_case(dtype, 1, 1, head_dim, page_size, [length], [1], seed=spot, v_transposed=transposed)
            plant(case, spot)
            out = _attend(case, 1, 1, head_dim, 1.0, window, length)
            value = case["vs"][0][spot, 0].float()
            assert (out[0].float().cpu() - value).abs().max() < 2e-2, (window, spot)
    # a key just outside the window must not be seen, nor one after the query
    for spot, q_len in ((length - 100 - 1, 1), (length - 1, 2)):
        case = _paged_case(dtype, 1, 1, head_dim, page_size, [length], [q_len], seed=5, v_transposed=transposed)
        plant(case, spot)  # `ks` is not changed: the plain model never sees that key
        out = _attend(case, 1, 1, head_dim, 1.0, 100, length)
        expected = _attention_expected(case, 1.0, 100)
        rows = slice(0, 1)  # the first query (position length - q_len) must not see the planted key
        assert np.abs(out.double().cpu().numpy() - expected)[rows].max() < _tol(dtype, 2)


def test_paged_attention_long_context_in_many_key_ranges():
    """One token over 9,000 keys of one head: the matrix-core kernel cuts them into more
    ranges than for short contexts; a planted key in the first, a middle and the last
    range is found, and an unplanted case matches the plain model."""
    from mini_infer_amd import ops

    head_dim, page_size, length = 128, 16, 9000
    assert min(32, ops.attention_splits(1, length, target=256, min_keys=128)) == 32
    for spot in (3, 4500, 8999):
        case = _paged_case(torch.bfloat16, 4, 1, head_dim, page_size, [length], [1], seed=spot, v_transposed=True)
        q = case["qs"][0][0, 2].float()  # the third of the four heads that share the keys
        page = case["block_table"][0, spot // page_size].item()
        case["k_pages"][page, 0, spot % page_size] = (q * 2.0).bfloat16().to(DEV)
        out = _attend(case, 4, 1, head_dim, 1.0, None, length)
        value = case["vs"][0][spot, 0].float()
        assert (out[0, 2 * head_dim : 3 * head_dim].float().cpu() - value).abs().max() < 2e-2, spot
    case = _paged_case(torch.bfloat16, 4, 1, head_dim, page_size, [length], [1], seed=11, v_transposed=True)
    out = _attend(case, 4, 1, head_dim, 0.05, None, length)
    expected = _attention_expected(case, 0.05, None)
    assert np.abs(out.double().cpu().numpy() - expected).max() < _tol(torch.bfloat16, 2)


@pytest.mark.parametrize(
    "q_heads,kv_heads,head_dim,lengths",
    [(32, 8, 128, [3000]), (6, 2, 64, [700, 2049]), (3, 1, 32, [517]), (32, 8, 128, [2100, 2500, 3000, 2048, 4000, 2222, 3100, 2900]),
     (6, 2, 64, [700, 2049, 333, 900, 1200, 800, 650, 1500, 400, 512, 2000])],
)
def test_output_projection_from_uncombined_key_ranges(q_heads, kv_heads, head_dim, lengths):
    """A few single tokens: the attention leaves its key ranges uncombined and the output
    projection combines them on its way; the same numbers as combining first."""
    from mini_infer_amd import ops

    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, 16, lengths, [1] * len(lengths), seed=41,
                       v_transposed=True)
    args = (case["q"], case["k_pages"], case["v_pages"], case["block_table"], case["token_request"],
            case["positions"], case["cu"], case["host_cu"])
    kwargs = dict(q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, scale=0.3, window=None,
                  max_seq_len=max(lengths), v_transposed=True)
    whole = ops.paged_attention(*args, **kwargs)
    pieces = ops.paged_attention(*args, **kwargs, combine=False)
    assert ops.attention_pieces_pay(1, q_heads, head_dim)
    assert isinstance(pieces, ops.AttentionPieces) and pieces.splits > 1 and pieces.tokens == len(lengths)
    assert (pieces.finish().float() - whole.float()).abs().max() < 2e-2
    for n in (q_heads * head_dim, 1000, 24):
        w = _rand(n, q_heads * head_dim, dtype=torch.bfloat16, seed=42, scale=0.1)
        assert torch.equal(ops.linear_from_attention(pieces, w), ops.linear(whole, w))
    # with nothing to combine, or more than single tokens, the attention comes back whole
    short = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, 16, [40], [1], seed=43, v_transposed=True)
    out = ops.paged_attention(short["q"], short["k_pages"], short["v_pages"], short["block_table"], short["token_request"],
                              short["positions"], short["cu"], short["host_cu"], q_heads=q_heads, kv_heads=kv_heads,
                              head_dim=head_dim, scale=0.3, window=None, max_seq_len=40, v_transposed=True, combine=False)
    assert isinstance(out, torch.Tensor)
    assert not ops.attention_pieces_pay(2, 32, 128) and not ops.attention_pieces_pay(1, 4, 48)


@pytest.mark.parametrize(
    "m,n,k,inter",
    [(8, 4096, 4096, 14336), (1, 4096, 4096, 14336), (16, 96, 64, 160), (7, 160, 96, 301), (13, 4128, 160, 40), (3, 32, 32, 5),
     (6, 1536, 1536, 520), (5, 1000, 512, 72), (16, 8200, 1024, 24)],
)
def test_product_add_and_norm_folded_into_two_products(m, n, k, inter):
    """`linear_add_norm` (product, add into the residual, norm but for the rows' factors) followed
    by `linear_swiglu` on its `ScaledRows`, against the four kernels they replace and against
    float64: the residual is bit-equal (the same rounded product added in float32), the
    activations agree as two bfloat16 roundings of the same numbers do."""
    from mini_infer_amd import ops

    x = _rand(m, k, dtype=torch.bfloat16, seed=51)
    w = _rand(n, k, dtype=torch.bfloat16, seed=52, scale=0.1)
    norm_w = (torch.rand(n, generator=torch.Generator().manual_seed(53)) + 0.5).bfloat16().to(DEV)
    gate_up = _rand(2 * inter, n, dtype=torch.bfloat16, seed=54, scale=0.08)
    residual0 = _rand(m, n, dtype=torch.float32, seed=55)
    eps = 3e-5

    apart_residual = residual0.clone()
    normed = ops.add_rmsnorm(ops.linear(x, w), apart_residual, norm_w, eps)
    apart = ops.linear_swiglu(normed, gate_up)

    residual = residual0.clone()
    rows = ops.linear_add_norm(ops.PendingProduct(x, w), residual, norm_w, eps)
    assert isinstance(rows, ops.ScaledRows) and rows.values.shape == (m, n) and rows.sumsq.shape[1] == m
    assert torch.equal(residual, apart_residual)
    # the pieces add up to the rows' sums of squares, and finish() is the norm's output
    exact_sumsq = (residual.double() ** 2).sum(dim=1)
    assert ((rows.sumsq.double().sum(dim=0) - exact_sumsq).abs() <= 1e-5 * exact_sumsq).all()
    exact_normed = residual.double() * torch.rsqrt(exact_sumsq / n + eps)[:, None] * norm_w.double()
    assert (rows.finish().double() - exact_normed).abs().max() < 2.0 ** -6 * float(exact_normed.abs().max())
    folded = ops.linear_swiglu(rows, gate_up)
    assert folded.shape == (m, inter)
    residual_off = residual0.clone()
    rows_off = ops.linear_add_norm(ops.PendingProduct(x, _off_the_cache_lines(w)), residual_off, norm_w, eps)
    assert torch.equal(residual_off, residual) and torch.equal(rows_off.values, rows.values)
    assert torch.equal(rows_off.sumsq, rows.sumsq)
    assert torch.equal(ops.linear_swiglu(rows, _off_the_cache_lines(gate_up)), folded)

    def activation(normed_rows):
        both = (normed_rows @ gate_up.double().T).bfloat16().double()
        return both[:, :inter] / (1 + torch.exp(-both[:, :inter])) * both[:, inter:]

    exact = activation(exact_normed)
    bound = 2.0 ** -5 * float(exact.abs().max()) + 1e-6
    assert (folded.double() - exact).abs().max() < bound
    assert (apart.double() - exact).abs().max() < bound  # (the yardstick: the four kernels are no closer)
    # rows that meet something else than that product are finished first: the same function
    assert ops.linear_swiglu(ops.ScaledRows(rows.values.float(), rows.sumsq, eps), gate_up.float()).shape == (m, inter)


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,lengths", [(32, 8, 128, [3000]), (6, 2, 64, [700]), (3, 1, 32, [517])])
def test_product_add_and_norm_from_uncombined_key_ranges(q_heads, kv_heads, head_dim, lengths):
    """The same fold with a single token's attention still in its key ranges: what
    `linear_from_attention` then `add_rmsnorm` give, bit for bit in the residual."""
    from mini_infer_amd import ops

    case = _paged_case(torch.bfloat16, q_heads, kv_heads, head_dim, 16, lengths, [1] * len(lengths), seed=61,
                       v_transposed=True)
    pieces = ops.paged_attention(
        case["q"], case["k_pages"], case["v_pages"], case["block_table"], case["token_request"], case["positions"],
        case["cu"], case["host_cu"], q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, scale=0.3, window=None,
        max_seq_len=max(lengths), v_transposed=True, combine=False)
    assert isinstance(pieces, ops.AttentionPieces)
    k, n = q_heads * head_dim, 4096 if head_dim == 128 else 200
    w = _rand(n, k, dtype=torch.bfloat16, seed=62, scale=0.1)
    norm_w = (torch.rand(n, generator=torch.Generator().manual_seed(63)) + 0.5).bfloat16().to(DEV)
    residual0 = _rand(len(lengths), n, dtype=torch.float32, seed=64)
    apart_residual, residual = residual0.clone(), residual0.clone()
    normed = ops.add_rmsnorm(ops.linear_from_attention(pieces, w), apart_residual, norm_w, 1e-5)
    rows = ops.linear_add_norm(ops.PendingProduct(pieces, w), residual, norm_w, 1e-5)
    assert torch.equal(residual, apart_residual)
    assert (rows.finish().float() - normed.float()).abs().max() <= 2.0 ** -6 * float(normed.float().abs().max())


@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize(
    "m,inter,hidden,q_heads,kv_heads,head_dim",
    [(8, 14336, 4096, 32, 8, 128), (1, 14336, 4096, 32, 8, 128), (16, 160, 96, 3, 1, 32), (5, 320, 160, 6, 2, 64), (3, 1536, 1536, 6, 2, 64)],
)
def test_down_product_add_and_norm_folded_into_the_next_q_k_v_product(v_transposed, m, inter, hidden, q_heads, kv_heads, head_dim):
    """`linear_add_norm` on a feed-forward's last product, then `qkv_rope_write` on its
    `ScaledRows`, against the three kernels they replace (product, add + norm, q|k|v with
    rotation and cache write): the residual bit for bit, queries, keys and values as two
    bfloat16 roundings of the same numbers agree, and against float64."""
    from mini_infer_amd import ops

    page_size, num_pages = 16, 5
    width = (q_heads + 2 * kv_heads) * head_dim
    act = _rand(m, inter, dtype=torch.bfloat16, seed=71)
    down = _rand(hidden, inter, dtype=torch.bfloat16, seed=72, scale=0.05)
    norm_w = (torch.rand(hidden, generator=torch.Generator().manual_seed(73)) + 0.5).bfloat16().to(DEV)
    qkv_w = _rand(width, hidden, dtype=torch.bfloat16, seed=74, scale=0.1)
    residual0 = _rand(m, hidden, dtype=torch.float32, seed=75)
    positions = torch.tensor([0, 1, 700, 5, 131071, 17, 18, 19, 3000, 2, 4, 6, 8, 10, 12, 14][:m], dtype=torch.int32, device=DEV)
    cos, sin = ops.rope_table(positions, torch.from_numpy(pl.inv_freq_default(head_dim, 500000.0)).to(DEV))
    slots = torch.tensor([40, 3, 17, 16, 0, 43, -1, 9, 22, 5, 6, 7, 30, 31, 32, 33][:m], dtype=torch.int32, device=DEV)
    eps = 2e-5

    def pages():
        k = torch.full((num_pages, kv_heads, page_size, head_dim), 7.0, dtype=torch.bfloat16, device=DEV)
        v_shape = (num_pages, kv_heads, head_dim, page_size) if v_transposed else k.shape
        return k, torch.full(v_shape, 7.0, dtype=torch.bfloat16, device=DEV)

    heads = dict(q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, v_transposed=v_transposed)
    apart_residual = residual0.clone()
    normed = ops.add_rmsnorm(ops.linear(act, down), apart_residual, norm_w, eps)
    k_apart, v_apart = pages()
    q_apart = ops.qkv_rope_write(normed, qkv_w, cos, sin, slots, k_apart, v_apart, **heads)

    residual = residual0.clone()
    rows = ops.linear_add_norm(ops.PendingProduct(act, down), residual, norm_w, eps)
    assert torch.equal(residual, apart_residual)
    assert ops.qkv_rope_write_takes(rows, qkv_w, head_dim, head_dim, False)
    k_fold, v_fold = pages()
    q_fold = ops.qkv_rope_write(rows, qkv_w, cos, sin, slots, k_fold, v_fold, **heads)

    # float64: the norm of the float32 residual the kernels left, the product rounded once, the rotation
    exact_sumsq = (residual.double() ** 2).sum(dim=1)
    exact_normed = residual.double() * torch.rsqrt(exact_sumsq / hidden + eps)[:, None] * norm_w.double()
    qkv = (exact_normed @ qkv_w.double().T).bfloat16().double().view(m, q_heads + 2 * kv_heads, head_dim)
    half = head_dim // 2
    c, s_ = cos.double()[:, None, :], sin.double()[:, None, :]
    rotated = torch.cat([qkv[..., :half] * c - qkv[..., half:] * s_, qkv[..., half:] * c + qkv[..., :half] * s_], dim=-1)
    exact_q = rotated[:, :q_heads].reshape(m, q_heads * head_dim)
    bound = 2.0 ** -5 * float(exact_q.abs().max()) + 1e-6
    assert (q_fold.double() - exact_q).abs().max() < bound
    assert (q_apart.double() - exact_q).abs().max() < bound  # (the yardstick: the three kernels are no closer)
    for row in range(m):
        slot = int(slots[row])
        if slot < 0:
            continue
        page, off = divmod(slot % (num_pages * page_size), page_size)
        exact_k = rotated[row, q_heads : q_heads + kv_heads]
        exact_v = qkv[row, q_heads + kv_heads :]
        got_v = v_fold[page, :, :, off] if v_transposed else v_fold[page, :, off]
        assert (k_fold[page, :, off].double() - exact_k).abs().max() < bound
        assert (got_v.double() - exact_v).abs().max() < bound
    # slots nobody wrote keep what they held, in both ways of running
    written = torch.zeros(num_pages * page_size, dtype=torch.bool, device=DEV)
    written[slots[slots >= 0].long()] = True
    untouched = ~written.view(num_pages, page_size)
    assert torch.all(k_fold.permute(0, 2, 1, 3)[untouched] == 7.0) and torch.all(k_apart.permute(0, 2, 1, 3)[untouched] == 7.0)
    # rows that meet a product without such a kernel are finished first: the same function
    many = ops.ScaledRows(rows.values.float(), rows.sumsq, eps)
    assert not ops.qkv_rope_write_takes(many, qkv_w.float(), head_dim, head_dim, False)


def test_kernels_refuse_what_they_do_not_take():
    from mini_infer_amd import ops
    from mini_infer_amd.exceptions import KernelShapeError

    for head_dim, message in ((25, "even"), (258, "at most 256")):
        case = _paged_case(torch.float32, 4, 2, head_dim, 4, [5], [1])
        with pytest.raises(KernelShapeError, match=message):
            _attend(case, 4, 2, head_dim, 1.0, None, 5)
    # transposed value pages belong to the matrix-core kernel, which takes bfloat16 only
    case = _paged_case(torch.float32, 4, 2, 32, 16, [5], [1], v_transposed=True)
    with pytest.raises(KernelShapeError, match="matrix-core"):
        _attend(case, 4, 2, 32, 1.0, None, 5)
    assert ops.mfma_attention_supported(torch.bfloat16, 128, 16)
    assert not ops.mfma_attention_supported(torch.bfloat16, 48, 16)
    assert not ops.mfma_attention_supported(torch.bfloat16, 128, 8)
    assert not ops.mfma_attention_supported(torch.float32, 128, 16)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ops.silu_mul(torch.zeros(2, 8))
    with pytest.raises(KernelShapeError):
        ops.add_rmsnorm(None, torch.zeros(2, 8, device=DEV), torch.ones(9, device=DEV), 1e-5)
    with pytest.raises(KernelShapeError):
        ops.gemm_f32(torch.zeros(2, 8, device=DEV), torch.zeros(3, 9, device=DEV))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens", [43, 150])  # (steps of fewer than 128 tokens do not look for pages)
@pytest.mark.parametrize("q_heads,kv_heads,dim,rotary,vdim,page,first", [(24, 8, 128, 128, 128, 16, 13), (3, 2, 72, 8, 24, 8, 8),
                                                                       (2, 1, 264, 256, 36, 8, 3), (5, 5, 8, 0, 4, 16, 0)])
def test_portions_that_fill_pages_write_what_single_tokens_write(dtype, tokens, q_heads, kv_heads, dim, rotary, vdim, page, first):
    """A page of transposed values that a step fills in order is written a dim's row at once, the others an element at a
    time; and a head by a part of a wave.  Token by token no page is filled: the same bits."""
    from mini_infer_amd import ops

    q_width, k_width, v_width = q_heads * dim, kv_heads * dim, kv_heads * vdim
    rows = _rand(tokens, q_width + k_width + v_width, dtype=dtype, seed=3)
    angles, other = _rand(tokens, rotary // 2, seed=4), _rand(tokens, v_width, dtype=dtype, seed=5)
    q_weight, k_weight, mix = _rand(q_width, seed=6), _rand(k_width, seed=7), torch.tensor([0.3], device=DEV)
    slots = torch.arange(first, first + tokens, dtype=torch.int32, device=DEV)
    slots[20] = -1  # a row that writes nowhere: its page is not filled
    made = []
    for step in (tokens, 1):
        left = []
        for op in range(2):
            qkv = rows.clone()
            k_pages = torch.zeros(1 + (first + tokens) // page, kv_heads, page, dim, dtype=dtype, device=DEV)
            v_pages = torch.zeros(1 + (first + tokens) // page, kv_heads, vdim, page, dtype=dtype, device=DEV)
            for t in range(0, tokens, step):
                part = slice(t, t + step)
                if op == 0:
                    ops.head_norm_rope_kv_write(qkv[part], angles[part].cos(), angles[part].sin(), slots[part].contiguous(), k_pages, v_pages,
                                                q_weight[:dim].contiguous(), k_weight[:dim].contiguous(), 1e-5, q_heads=q_heads, kv_heads=kv_heads,
                                                head_dim=dim, rotary_dim=rotary, v_head_dim=vdim, v_transposed=True)
                else:
                    ops.qkv_norm_write(qkv[part], q_weight, k_weight, slots[part].contiguous(), k_pages, v_pages, q_width=q_width,
                                       kv_heads=kv_heads, head_dim=dim, v_head_dim=vdim, eps=1e-5, other_values=other[part], mix=mix,
                                       v_transposed=True)
            left += [qkv, k_pages, v_pages]
        made.append(left)
    for whole, single in zip(*made):
        assert torch.equal(whole, single)
    normed = rows[:, :q_width].double().view(tokens, q_heads, dim)
    normed = normed / torch.sqrt((normed * normed).mean(-1, keepdim=True) + 1e-5) * q_weight[:dim].double()
    turned = normed.clone()
    if rotary:
        cos, sin = angles.double().cos()[:, None], angles.double().sin()[:, None]
        lo, hi = normed[..., : rotary // 2], normed[..., rotary // 2 : rotary]
        turned[..., :rotary] = torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), -1)
    got = made[0][0][:, :q_width].double().view(tokens, q_heads, dim)
    # one rounding to the element type, and a few float32 roundings before it
    assert (got - turned).abs().max() <= (2.0 ** -8 if dtype == torch.bfloat16 else 1e-6) * turned.abs().max()


@pytest.mark.parametrize("heads,dim,rot,vdim,v_width,page,spare", [(5, 128, 64, 128, 128, 16, 8), (32, 16, 16, 12, 32, 8, 0), (3, 20, 12, 20, 32, 16, 0),
                                                                   (4, 64, 0, 64, 64, 16, 3), (1, 24, 8, 7, 32, 4, 0)])
@pytest.mark.parametrize("apart", [False, True])
def test_latent_keys_and_values_of_a_step_in_pages(heads, dim, rot, vdim, v_width, page, spare, apart):
    """Pages written whole, zeros where no token lies; queries rotated in place where rows allow it, else beside."""
    from mini_infer_amd import ops

    lengths, width = [1, 33, 16, 40], dim + rot
    tokens = sum(lengths)
    held = _rand(tokens, rot + 8, dtype=torch.bfloat16, seed=2)
    proj = _rand(tokens, heads * width + (0 if apart else rot) + spare, dtype=torch.bfloat16, seed=3)
    shared = held[:, 8:] if apart else proj[:, heads * width : heads * width + rot]
    before, shared = proj.clone(), shared.clone()
    k_up, v_up = _rand(tokens, heads * dim, dtype=torch.bfloat16, seed=4), _rand(tokens, heads * vdim + spare, dtype=torch.bfloat16, seed=5)[:, : heads * vdim]
    angles = _rand(tokens, rot // 2, seed=6)
    first, count, start = [], [], 0
    for n in lengths:
        for at in range(0, n, page):
            first.append(start + at), count.append(min(page, n - at))
        start += n
    k_pages = torch.full((len(first), heads, page, width), float("nan"), dtype=torch.bfloat16, device=DEV)
    v_pages = torch.full((len(first), heads, v_width, page), float("nan"), dtype=torch.bfloat16, device=DEV)
    ints = [torch.tensor(x, dtype=torch.int32, device=DEV) for x in (first, count)]
    queries = ops.latent_expand_pages(proj, k_up, v_up, angles.cos(), angles.sin(), k_pages, v_pages, *ints, heads=heads, dim=dim, rot=rot,
                                      vdim=vdim, r_col=8 if apart else heads * width, down=held if apart else None)

    def turned(x):  # [..., rot], pairs side by side
        pairs = x.float().unflatten(-1, (rot // 2, 2))
        cos, sin = (f().view(tokens, *[1] * (pairs.dim() - 3), rot // 2) for f in (angles.cos, angles.sin))
        return torch.stack((pairs[..., 0] * cos - pairs[..., 1] * sin, pairs[..., 1] * cos + pairs[..., 0] * sin), -1).flatten(-2)

    q = before[:, : heads * width].view(tokens, heads, width)
    want_q = torch.cat((q[..., :dim].float(), turned(q[..., dim:])), -1)
    want_k = torch.cat((k_up.view(tokens, heads, dim).float(), turned(shared)[:, None].expand(tokens, heads, rot)), -1)
    got_q = queries[:, : heads * width].view(tokens, heads, width).float()
    # (one rounding to bfloat16, of sums of two products)
    assert ((got_q - want_q).abs() <= 2.0 ** -8 * want_q.abs() + 1e-6).all()
    assert torch.equal(proj[:, heads * width :], before[:, heads * width :])
    for p, (t, n) in enumerate(zip(first, count)):
        got_k, got_v = k_pages[p].transpose(0, 1).float(), v_pages[p].permute(2, 0, 1)
        assert ((got_k[:n] - want_k[t : t + n]).abs() <= 2.0 ** -8 * want_k[t : t + n].abs() + 1e-6).all() and (got_k[n:] == 0).all()
        assert torch.equal(got_v[:n, :, :vdim], v_up[t : t + n].view(n, heads, vdim))
        assert (got_v[n:] == 0).all() and (got_v[:, :, vdim:] == 0).all()


@pytest.mark.parametrize("q_heads,kv_heads,dim,page,window,lengths,contexts", [
    (32, 8, 64, 16, None, [131], [0]), (24, 8, 128, 16, 37, [100, 66, 1, 33], [0, 50, 200, 7]), (40, 2, 64, 32, None, [130, 61], [3, 0]),
    (16, 16, 64, 16, 1, [300], [70]), (32, 2, 64, 48, 100, [257], [1000])])
def test_prompt_attention_float32(q_heads, kv_heads, dim, page, window, lengths, contexts):
    """Row tiles across requests, groups that leave rows idle or need several blocks, windows, keys past the last one that are
    no numbers; against the plain kernel."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import library

    tokens = sum(lengths)
    assert library.load().mi_attn_prompt_f32_blocks(tokens, q_heads, kv_heads, dim, page) >= 256 and tokens >= 32 * len(lengths)
    pages_of = [-(-(n + c) // page) for n, c in zip(lengths, contexts)]
    order = torch.randperm(sum(pages_of), generator=torch.Generator().manual_seed(1)).int()
    table = torch.zeros(len(lengths), max(pages_of), dtype=torch.int32)
    at = 0
    k_pages, v_pages = (_rand(sum(pages_of), kv_heads, page, dim, seed=s) for s in (2, 3))
    for b, count in enumerate(pages_of):
        table[b, :count] = order[at : at + count]
        at += count
        past = lengths[b] + contexts[b] - (count - 1) * page
        for pages in (k_pages, v_pages):
            pages[int(table[b, count - 1]), :, past:] = float("nan")
    last = int(table[-1, (lengths[-1] + contexts[-1] - 1) // page]), (lengths[-1] + contexts[-1] - 1) % page
    v_pages[last[0], :, last[1]] = float("inf")  # the last token's own value: the tokens before it do not see it
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    requests = ints([b for b, n in enumerate(lengths) for _ in range(n)])
    positions = ints([c + i for n, c in zip(lengths, contexts) for i in range(n)])
    cu = [0, *torch.tensor(lengths).cumsum(0).tolist()]
    q = _rand(tokens, q_heads * dim + 4, seed=4)
    got, plain = (
        ops.paged_attention(q, k_pages, v_pages, table.to(DEV), requests, positions, ints(cu), cu, q_heads=q_heads, kv_heads=kv_heads,
                            head_dim=dim, scale=dim ** -0.5, window=window, max_seq_len=max(n + c for n, c in zip(lengths, contexts)),
                            force_plain=plain)
        for plain in (False, True))
    assert torch.isinf(got[-1]).all() and torch.isinf(plain[-1]).all()
    # both round a result once; the plain kernel also each weight (weights sum to one) and, with cut keys, each part
    most = float(v_pages[torch.isfinite(v_pages)].abs().max())
    assert (got[:-1] - plain[:-1]).abs().max() <= 4 * 2.0 ** -24 * most


@pytest.mark.parametrize("q_heads,kv_heads,dim,requests,longest,window", [
    (24, 8, 128, 90, 128, None), (24, 8, 128, 110, 128, None), (24, 8, 128, 110, 130, None), (6, 3, 80, 300, 300, 65), (4, 4, 64, 2, 65, None),
    (8, 8, 64, 260, 20, None)])
def test_decoded_tokens_attention_float32(q_heads, kv_heads, dim, requests, longest, window):
    """On both sides of the line between one wave and four a block; contexts of 1, 64 and 65 keys, which leave waves idle, and the
    longest, in one launch; in 64 bits."""
    from mini_infer_amd import ops

    page = 16
    keys = [(1, 64, 65, longest)[b % 4] if longest >= 65 else 1 + b % longest for b in range(requests)]
    keys = [min(n, longest) for n in keys]
    blocks = max(-(-n // page) for n in keys)
    k_pages, v_pages = (_rand(requests * blocks, kv_heads, page, dim, seed=s) for s in (2, 3))
    table = torch.randperm(requests * blocks, generator=torch.Generator().manual_seed(1)).int().view(requests, blocks).to(DEV)
    q = _rand(requests, q_heads * dim, seed=4)
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    cu = list(range(requests + 1))
    got = ops.paged_attention(q, k_pages, v_pages, table, ints(cu[:-1]), ints([n - 1 for n in keys]), ints(cu), cu, q_heads=q_heads,
                              kv_heads=kv_heads, head_dim=dim, scale=dim ** -0.5, window=window, max_seq_len=max(keys))
    seen = torch.arange(blocks * page, device=DEV)[None] < ints(keys)[:, None]
    if window is not None:
        seen &= torch.arange(blocks * page, device=DEV)[None] >= ints(keys)[:, None] - window
    k, v = (pages[table.long()].transpose(2, 3).reshape(requests, -1, kv_heads, dim).repeat_interleave(q_heads // kv_heads, 2).double() for pages in (k_pages, v_pages))
    scores = (q.view(requests, 1, q_heads, dim).double() * k).sum(-1) * dim ** -0.5
    weights = torch.softmax(scores.masked_fill(~seen[..., None], float("-inf")), 1)
    want = (weights[..., None] * v).sum(1).flatten(1)
    # a weight and the result are rounded once each (weights sum to one)
    assert (got.double() - want).abs().max() <= 3 * 2.0 ** -24 * float(v_pages.abs().max())


@pytest.mark.parametrize("q_heads,kv_heads,dim,lengths,contexts,launches", [
    (24, 8, 128, [1, 1, 1, 200], [700, 0, 64, 30], ["tiles", "plain"]), (8, 8, 64, [1] * 5 + [300, 290], [90] * 7, ["tiles", "plain"]),
    (24, 8, 128, [1, 1, 60], [70, 3, 0], ["plain"]), (8, 8, 64, [520] + [1] * 9, [20] * 10, ["plain"]), (24, 8, 128, [170], [9], ["tiles"])])
def test_mixed_step_attention_float32(monkeypatch, q_heads, kv_heads, dim, lengths, contexts, launches):
    """Leading single tokens apart from the portions, where those go in tiles; all in one plain launch else.  In 64 bits."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import library

    lib, taken = library.load(), []
    for kind, name in (("tiles", "mi_attn_prompt_f32"), ("plain", "mi_attn_generic")):
        entry = getattr(lib, name)
        monkeypatch.setattr(lib, name, lambda *args, kind=kind, entry=entry: (taken.append(kind), entry(*args))[1])
    page, keys = 16, [n + c for n, c in zip(lengths, contexts)]
    blocks = max(-(-n // page) for n in keys)
    k_pages, v_pages = (_rand(len(lengths) * blocks, kv_heads, page, dim, seed=s) for s in (2, 3))
    table = torch.randperm(len(lengths) * blocks, generator=torch.Generator().manual_seed(1)).int().view(-1, blocks).to(DEV)
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    cu = [0, *torch.tensor(lengths).cumsum(0).tolist()]
    q = _rand(cu[-1], q_heads * dim + 4, seed=4)[:, : q_heads * dim]
    positions = [c + i for n, c in zip(lengths, contexts) for i in range(n)]
    got = ops.paged_attention(q, k_pages, v_pages, table, ints([b for b, n in enumerate(lengths) for _ in range(n)]), ints(positions), ints(cu), cu,
                              q_heads=q_heads, kv_heads=kv_heads, head_dim=dim, scale=dim ** -0.5, window=None, max_seq_len=max(keys))
    assert taken == launches
    for b, n in enumerate(lengths):
        k, v = (pages[table[b].long()].transpose(1, 2).reshape(-1, kv_heads, dim).repeat_interleave(q_heads // kv_heads, 1).double() for pages in (k_pages, v_pages))
        rows = slice(cu[b], cu[b + 1])
        scores = torch.matmul(q[rows].view(n, q_heads, dim).double().transpose(0, 1), k.permute(1, 2, 0).contiguous()) * dim ** -0.5
        scores.masked_fill_(torch.arange(k.shape[0], device=DEV)[None] > ints(positions[rows])[:, None], float("-inf"))
        want = torch.matmul(torch.softmax(scores, -1), v.transpose(0, 1).contiguous()).transpose(0, 1).flatten(1)
        # a weight and the result are rounded once each (weights sum to one), and each part where keys are cut
        assert (got[rows].double() - want).abs().max() <= 4 * 2.0 ** -24 * float(v_pages.abs().max())


@pytest.mark.parametrize("tokens,plain", [(520, False), (520, True), (1, True)])
@pytest.mark.parametrize("low", [[16], [32, 33], list(range(64, 128)), list(range(100, 300))])
def test_scores_of_minus_infinity_have_no_weight_float32(tokens, plain, low):
    """Keys whose scores are -inf (an infinite element), also where a tile of keys, or all that a wave has seen so far, has no
    others: left out, as a score that is very low is."""
    from mini_infer_amd import ops

    q_heads, kv_heads, dim, page, length = 8, 8, 64, 16, 520 if tokens > 1 else 500
    k_pages, v_pages = (_rand(-(-length // page), kv_heads, page, dim, seed=s) for s in (2, 3))
    flat = k_pages.transpose(1, 2).reshape(-1, kv_heads, dim)
    flat[low, :, 0] = float("inf")
    k_pages = flat.view(-1, page, kv_heads, dim).transpose(1, 2).contiguous()
    q = _rand(tokens, q_heads * dim, seed=4)
    q.view(tokens, q_heads, dim)[:, :, 0] = -1.0 - q.view(tokens, q_heads, dim)[:, :, 0].abs()
    first = 0 if tokens > 1 else length - 1
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    got = ops.paged_attention(q, k_pages, v_pages, torch.arange(len(k_pages), dtype=torch.int32, device=DEV)[None], ints([0] * tokens),
                              ints([first + i for i in range(tokens)]), ints([0, tokens]), [0, tokens], q_heads=q_heads, kv_heads=kv_heads, head_dim=dim,
                              scale=dim ** -0.5, window=None, max_seq_len=first + tokens, force_plain=plain)
    v = v_pages.transpose(1, 2).reshape(-1, kv_heads, dim).double()
    scores = torch.matmul(q.view(tokens, q_heads, dim).double().transpose(0, 1), flat.double().permute(1, 2, 0).contiguous()) * dim ** -0.5
    scores.masked_fill_(torch.arange(len(flat), device=DEV)[None] > (first + torch.arange(tokens, device=DEV))[:, None], float("-inf"))
    want = torch.matmul(torch.softmax(scores, -1), v.transpose(0, 1).contiguous()).transpose(0, 1).flatten(1)
    assert want.isfinite().all() and got.isfinite().all()
    assert (got.double() - want).abs().max() <= 4 * 2.0 ** -24 * float(v_pages.abs().max())


@pytest.mark.parametrize("m", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("n,k", [(40, 4), (33, 36), (8200, 100), (100, 2052), (17, 63), (8193, 258)])
def test_few_rows_of_gemm_f32_off_whole_lines(m, n, k):
    """Rows of W that end inside a line or start off one: loads by 16 bytes and by single values, whose masked parts (infinite
    first values here) add nothing; the bits of 16-byte rows, of single values and of many rows are the same."""
    from mini_infer_amd import ops

    a, w = _rand(m, k, seed=31), _rand(n, k, seed=32)
    a[:, 0], w[:, 0] = 1.0, float("inf")  # (every sum is infinite, so an addend of 0 * inf would show as NaN)
    assert torch.isinf(ops.gemm_f32(a, w)).all()
    w[:, 0] = 0.5
    out = ops.gemm_f32(a, w)
    exact = a.double() @ w.double().T
    assert ((out.double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 1e-12 * math.sqrt(k)).all()
    for before_a, before_w in ((4, 4), (0, 4), (4, 0), (1, 4), (4, 3)):
        off_a, off_w = torch.full((m, k + 4), 3.0, device=DEV), torch.full((n, k + 4), 5.0, device=DEV)
        off_a, off_w = off_a[:, before_a : before_a + k], off_w[:, before_w : before_w + k]
        off_a.copy_(a), off_w.copy_(w)
        assert torch.equal(ops.gemm_f32(off_a, off_w), out), (before_a, before_w)
    many = torch.cat([a, torch.ones(70, k, device=DEV)])
    assert torch.equal(ops.gemm_f32(many, w)[:m], out)


@pytest.mark.parametrize("tokens,width", [(1025, 512), (2049, 512), (2051, 6000)])
def test_router_block_sizes_give_the_same_bits(tokens, width):
    """Sixteen, ten and four waves a block, by how many blocks there are and how much LDS one takes."""
    from mini_infer_amd import ops

    x, router = _rand(tokens, width, dtype=torch.bfloat16, seed=51), _rand(10, width, seed=52, scale=0.05)
    chosen, weights, _ = ops.route_top_k(x, router, None, None, top=3, route_scale=1.0)
    for at in range(0, tokens, 500):
        some, their, _ = ops.route_top_k(x[at : at + 500], router, None, None, top=3, route_scale=1.0)
        assert torch.equal(chosen[at : at + 500], some) and torch.equal(weights[at : at + 500], their)
    want = torch.softmax(x.double() @ router.double().T, 1).gather(1, chosen.long())
    assert ((weights.double() - want).abs() <= 1e-5 * want).all()  # float32 sums of `width` products, and exponentials of them


@pytest.mark.parametrize("groups,group,period", [(5, 63, 63), (3, 1023, 3069), (2, 1025, 1025), (3, 2050, 6150), (1, 4100, 41), (7, 9, 3), (2, 4096, 8192)])
@pytest.mark.parametrize("gate_first", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_readout_norm_groups_of_any_size(groups, group, period, gate_first, dtype):
    """Groups that the threads hold at once and that they do not, by fours and by single columns, weights that wrap inside a group."""
    from mini_infer_amd import ops

    width = groups * group
    o, gate, weight = _rand(5, width, seed=61), _rand(5, width + 1, dtype=dtype, seed=62)[:, 1:], 1 + 0.2 * _rand(period, seed=63)
    got = ops.readout_gate_norm(o, gate, weight, group_width=group, gate_first=gate_first, eps=1e-5).double()
    silu = gate.double() * torch.sigmoid(gate.double())
    y = (o.double() * silu if gate_first else o.double()).view(5, groups, group)
    y = (y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-5)).view(5, width) * weight.double().repeat(width // period)
    want = y if gate_first else y * silu
    # one rounding to the element type, and a few float32 roundings before it
    assert ((got - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 1e-5) * want.abs() + 1e-6).all()


@pytest.mark.parametrize("heads,dim,rot,vdim,spare", [(5, 128, 64, 128, 8), (3, 20, 12, 20, 0), (4, 64, 0, 30, 3), (2, 24, 8, 32, 1)])
@pytest.mark.parametrize("apart", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_latent_heads_as_one_row_a_token(heads, dim, rot, vdim, spare, apart, dtype):
    from mini_infer_amd import ops

    tokens, width = 37, dim + rot
    held = _rand(tokens, spare + rot, dtype=dtype, seed=2)
    proj = _rand(tokens, heads * width + (0 if apart else spare + rot), dtype=dtype, seed=1)
    before, shared = proj.clone(), held[:, spare:] if apart else proj[:, heads * width + spare :]
    k_up, v_up = _rand(tokens, heads * dim, dtype=dtype, seed=3), _rand(tokens, heads * vdim, dtype=dtype, seed=4)
    angles = _rand(tokens, rot // 2, seed=5)
    got = ops.latent_expand(proj, k_up, v_up, angles.cos(), angles.sin(), heads=heads, dim=dim, rot=rot, vdim=vdim,
                            r_col=spare if apart else heads * width + spare, down=held if apart else None)
    assert torch.equal(proj, before) and got.shape == (tokens, 3 * heads * width)

    def turned(x):  # [tokens, heads, rot], pairs side by side
        pairs, cos, sin = x.double().unflatten(-1, (rot // 2, 2)), angles.double().cos()[:, None], angles.double().sin()[:, None]
        return torch.stack((pairs[..., 0] * cos - pairs[..., 1] * sin, pairs[..., 1] * cos + pairs[..., 0] * sin), -1).flatten(-2)

    q, k, v = got.double().view(tokens, 3, heads, width).unbind(1)
    want_q = before[:, : heads * width].double().view(tokens, heads, width)
    assert torch.equal(q[..., :dim], want_q[..., :dim]) and torch.equal(k[..., :dim], k_up.double().view(tokens, heads, dim))
    assert torch.equal(v[..., :vdim], v_up.double().view(tokens, heads, vdim)) and (v[..., vdim:] == 0).all()
    for made, source in ((q, want_q[..., dim:]), (k, shared[:, None].expand(tokens, heads, rot))):
        want = turned(source)
        # one rounding to the element type, of sums of two float32 products with float32 sines
        assert ((made[..., dim:] - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 1e-6) * (want.abs() + 1)).all()


@pytest.mark.parametrize("dim,spare", [(128, 0), (20, 0), (128, 3)])
def test_latent_queries_are_rotated_in_place_only_when_asked_to(dim, spare):
    """The same bits either way; without `in_place` the projections stay as they are, whatever their alignment."""
    from mini_infer_amd import ops

    heads, rot, tokens, page = 3, 64, 21, 16
    proj = _rand(tokens, heads * (dim + rot) + rot + spare, dtype=torch.bfloat16, seed=1)[:, spare:]
    before, angles = proj.clone(), _rand(tokens, rot // 2, seed=5)
    k_up, v_up = (_rand(tokens, heads * dim, dtype=torch.bfloat16, seed=s) for s in (3, 4))
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    made = []
    for in_place in (False, True):
        k_pages, v_pages = (torch.zeros(2, heads, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((page, dim + rot), (dim, page)))
        rows = ops.latent_expand_pages(proj, k_up, v_up, angles.cos(), angles.sin(), k_pages, v_pages, ints([0, 16]), ints([16, 5]), heads=heads,
                                       dim=dim, rot=rot, vdim=dim, r_col=heads * (dim + rot), in_place=in_place)
        made.append((rows[:, : heads * (dim + rot)].clone(), k_pages, v_pages))
        if not in_place:
            assert torch.equal(proj, before)
    assert all(torch.equal(a, b) for a, b in zip(*made))


@pytest.mark.parametrize("m,hidden,heads,kv_heads,head_dim", [(1, 256, 2, 1, 16), (3, 2048, 6, 2, 64), (4, 8192, 3, 1, 32), (8, 1024, 4, 4, 128), (2, 64, 3, 0, 48)])
@pytest.mark.parametrize("transposed", [False, True])
def test_float32_rows_projected_rotated_and_written_as_one(m, hidden, heads, kv_heads, head_dim, transposed):
    """Against `linear` and `rope_kv_write`: the same bits."""
    from mini_infer_amd import ops

    torch.manual_seed(m + hidden)
    page, pages = 16, 3
    x = torch.randn(m, hidden, device="cuda")
    w = torch.randn((heads + 2 * kv_heads) * head_dim, hidden, device="cuda") / hidden ** 0.5
    angle = torch.rand(m, head_dim // 2, device="cuda") * 6
    cos, sin = angle.cos(), angle.sin()
    slots = torch.tensor([5, 17, -1, 33, 16, 47, 0, 31][:m], dtype=torch.int32, device="cuda")
    sizes = (pages, max(kv_heads, 1), page, head_dim)
    caches = [[torch.zeros(sizes, device="cuda"), torch.zeros(sizes[:2] + (head_dim, page) if transposed else sizes, device="cuda")] for _ in range(3)]
    names = dict(q_heads=heads, kv_heads=kv_heads, head_dim=head_dim, v_transposed=transposed)
    where = [(slots, *c) if kv_heads else (None, None, None) for c in caches]
    assert ops.qkv_rope_write_f32_takes(x, w, head_dim, head_dim, False)
    apart = ops.rope_kv_write(ops.linear(x, w), cos, sin, *where[0], rotary_dim=head_dim, **names)[:, : heads * head_dim]
    one = ops.qkv_rope_write_f32(x, w, cos, sin, *where[1], **names)
    assert torch.equal(one, apart) and all(torch.equal(ours, theirs) for ours, theirs in zip(caches[1], caches[0]))


@pytest.mark.parametrize("m,hidden,heads,kv_heads,head_dim,page", [
    (33, 3072, 24, 8, 128, 16), (271, 3072, 24, 8, 128, 16), (97, 2048, 6, 1, 96, 8), (350, 256, 6, 2, 64, 16), (1030, 128, 3, 3, 32, 32),
    (513, 64, 5, 1, 16, 12), (700, 128, 4, 0, 48, 16), (321, 192, 2, 2, 256, 4),
])
@pytest.mark.parametrize("transposed", [False, True])
def test_many_rows_projected_rotated_and_written_as_one(m, hidden, heads, kv_heads, head_dim, page, transposed):
    """In every tile that the kernel may take, against the same tile's plain product and `rope_kv_write`: the same bits."""
    from mini_infer_amd import ops
    from mini_infer_amd.exceptions import KernelShapeError
    from mini_infer_amd.ops import kernels, library

    torch.manual_seed(m + hidden)
    x = torch.randn(m, hidden, device="cuda").bfloat16()
    n = (heads + 2 * kv_heads) * head_dim
    w = (torch.randn(n, hidden, device="cuda") / hidden ** 0.5).bfloat16()
    angle = torch.rand(m, head_dim // 2, device="cuda") * 6
    cos, sin = angle.cos(), angle.sin()
    # single slots, rows that are not written, a run from the middle of a page on and one that begins a page
    pages = 2 * (m // page) + 20
    free = torch.randperm(9 * page)[:9].tolist()
    run = list(range(10 * page + 5, 10 * page + 5 + (m - 11) // 2))
    slots = free + [-1, -1] + run
    begin = (slots[-1] // page + 2) * page
    slots = torch.tensor(slots + list(range(begin, begin + m - len(slots))), dtype=torch.int32, device="cuda")
    assert slots.max() < pages * page and slots.unique().numel() == m - 1
    sizes = (pages, max(kv_heads, 1), page, head_dim)
    names = dict(q_heads=heads, kv_heads=kv_heads, head_dim=head_dim, v_transposed=transposed)

    def caches():
        return [torch.zeros(sizes, device="cuda", dtype=torch.bfloat16),
                torch.zeros(sizes[:2] + (head_dim, page) if transposed else sizes, device="cuda", dtype=torch.bfloat16)]

    def check(product, plan, form=-1):
        theirs, ours = caches(), caches()
        where = [(slots, *c) if kv_heads else (None, None, None) for c in (theirs, ours)]
        apart = ops.rope_kv_write(product, cos, sin, *where[0], rotary_dim=head_dim, **names)[:, : heads * head_dim]
        if form < 0:
            one = ops.qkv_rope_write_many(x, w, cos, sin, *where[1], plan=plan, **names)
        else:  # all tiles of that form
            one = torch.empty(m, heads * head_dim, dtype=torch.bfloat16, device="cuda")
            pointers = [None if t is None else t.data_ptr() for t in where[1]]
            library.check(library.load().mi_gemm_turns_rope(
                x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), one.data_ptr(), one.stride(0), cos.data_ptr(), sin.data_ptr(), *pointers, m, hidden,
                heads, kv_heads, head_dim, page, pages, int(transposed), form, torch.cuda.current_stream().cuda_stream))
        assert torch.equal(one, apart) and torch.equal(ours[0], theirs[0]) and torch.equal(ours[1], theirs[1])

    if m > 320:
        form = 0
        while library.load().mi_gemm_turns_rows(form):
            check(kernels._turns(0, x, w, n), -1, form)
            form += 1
    else:
        shape = 0
        while kernels.tile_size(shape)[0]:
            plain = kernels._tiles(0, x, w, torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), n, shape, 1)
            check(plain, shape)
            shape += 1
    plan = ops.qkv_rope_write_many_plan(x, w, head_dim, head_dim, False)
    assert m <= 320 or plan is None or plan == -1
    if m > 320 and plan is not None or m <= 320 and kernels.tiles_for(m, n, hidden, False):
        check(ops.linear(x, w), plan)
    with pytest.raises(KernelShapeError):
        ops.qkv_rope_write_many(x[:, ::2], w[:, ::2], cos, sin, None, None, None, plan=-1, **names)
    assert ops.qkv_rope_write_many_plan(x, w, head_dim, head_dim, True) is None
    assert ops.qkv_rope_write_many_plan(x.float(), w.float(), head_dim, head_dim, False) is None


@pytest.mark.parametrize("m, k, heads, kv_heads, head_dim, how, kind", [
    (271, 3072, 24, 8, 128, {}, "tiles"), (97, 2048, 6, 1, 128, {}, "tiles"), (320, 768, 12, 12, 64, {}, "tiles"), (100, 2048, 16, 0, 64, {}, "tiles"),
    (400, 768, 12, 12, 64, {}, "turns"), (512, 2048, 16, 8, 128, {}, "turns"), (700, 1024, 16, 0, 64, {}, "turns"),
    (700, 1024, 16, 8, 64, {"steady": True}, "turns"), (400, 768, 12, 12, 64, {"in_pieces": True}, "turns"),
    (271, 3072, 24, 8, 128, {"steady": True}, None), (271, 3072, 24, 8, 128, {"in_pieces": True}, None), (32, 3072, 24, 8, 128, {}, None),
    (64, 8192, 4, 2, 64, {}, None), (330, 8192, 4, 2, 64, {}, None), (2060, 512, 64, 64, 128, {"steady": True}, None), (2060, 512, 64, 64, 128, {}, "turns"),
    (300, 96, 4, 2, 64, {}, None), (271, 3072, 24, 8, 128, {"interleaved": True}, None), (271, 3072, 24, 8, 128, {"rotary_dim": 64}, None),
    (271, 3072, 16, 8, 200, {}, None), (271, 3072, 24, 8, 128, {"off": True}, None)])
def test_which_projections_are_rotated_in_their_tiles(m, k, heads, kv_heads, head_dim, how, kind):
    """The plan from the public entry, and what it makes against the same tiles' plain product and `rope_kv_write`."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    n = (heads + 2 * kv_heads) * head_dim
    x, w = _rand(m, k, dtype=torch.bfloat16, seed=60), _rand(n, k, dtype=torch.bfloat16, seed=61, scale=k ** -0.5)
    angle = torch.rand(m, head_dim // 2, device="cuda") * 6
    cos, sin = angle.cos(), angle.sin()
    others = (cos, sin, torch.empty(9, device="cuda")[1:] if how.get("off") else None)
    plan = ops.qkv_rope_write_many_plan(x, w, head_dim, how.get("rotary_dim", head_dim), how.get("interleaved", False), how.get("steady", False),
                                        how.get("in_pieces", False), others)
    assert (kind is None) == (plan is None) and (kind is None or (kind == "turns") == (plan == -1))
    if plan is None:
        return
    product = kernels._turns(0, x, w, n) if plan < 0 else kernels._tiles(0, x, w, torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), n, plan, 1)
    slots = torch.randperm(m + 40, device="cuda").int()[:m].contiguous()
    made = []
    names = dict(q_heads=heads, kv_heads=kv_heads, head_dim=head_dim, v_transposed=True)
    for as_one in (False, True):
        pages = [torch.zeros(m // 16 + 4, max(kv_heads, 1), *shape, dtype=torch.bfloat16, device="cuda") for shape in ((16, head_dim), (head_dim, 16))]
        where = (slots, *pages) if kv_heads else (None, None, None)
        if as_one:
            queries = ops.qkv_rope_write_many(x, w, cos, sin, *where, plan=plan, **names)
        else:
            queries = ops.rope_kv_write(product, cos, sin, *where, rotary_dim=head_dim, **names)[:, : heads * head_dim]
        made.append([queries, *pages])
    assert all(torch.equal(a, b) for a, b in zip(*made))


LAUNCHES = ("mi_gemm_turns_rope", "mi_gemm_tiles_rope", "mi_gemm_f32_rope", "mi_gemm_turns_bf16", "mi_gemm_tiles_bf16", "mi_rope_kv_write")


@pytest.mark.parametrize("dtype, steady, rows, rotates", [
    (torch.float32, False, 1, "mi_gemm_f32_rope"), (torch.float32, False, 4, "mi_gemm_f32_rope"), (torch.float32, False, 5, "mi_gemm_f32_rope"),
    (torch.float32, False, 8, "mi_gemm_f32_rope"), (torch.float32, False, 9, "mi_rope_kv_write"), (torch.float32, False, 100, "mi_rope_kv_write"),
    (torch.bfloat16, False, 100, "mi_gemm_tiles_rope"), (torch.bfloat16, False, 320, "mi_gemm_tiles_rope"), (torch.bfloat16, False, 400, "mi_gemm_turns_rope"),
    (torch.bfloat16, True, 100, "mi_rope_kv_write"), (torch.bfloat16, True, 400, "mi_gemm_turns_rope")])
def test_what_a_models_step_launches(dtype, steady, rows, rotates, monkeypatch):
    """A prompt of so many tokens (up to 9: so many requests, a token each) through a small Llama: which kernel rotates and writes q|k|v, in every layer, and no product of a steady
    one in tiles of another order.  The logits against the same step where nothing is rotated in a product."""
    from mini_infer_amd import ModelRunner, StepEntry, ops
    from mini_infer_amd.models import architecture_for
    from mini_infer_amd.ops import kernels, library

    config = {"architectures": ["LlamaForCausalLM"], "num_hidden_layers": 2, "hidden_size": 512, "num_attention_heads": 8, "num_key_value_heads": 4,
              "head_dim": 64, "intermediate_size": 1024, "vocab_size": 256, "rope_theta": 10000.0, "rms_norm_eps": 1e-5, "tie_word_embeddings": False,
              "max_position_embeddings": 1024}
    arch = architecture_for(config)
    parsed = arch.parse_config(config)
    model = arch.make_model(parsed, dtype, "cuda:0")
    specs, generator = model.param_specs(), torch.Generator(device="cuda").manual_seed(7)
    model.load_params(lambda name: (torch.randn(specs[name].shape, generator=generator, device="cuda") * (1.0 if len(specs[name].shape) == 1 else 0.05)).to(
        torch.float32 if specs[name].dtype == "float32" else dtype))
    for block in model.blocks:
        for part in block.parts():
            part.steady = steady
    lib, taken = library.load(), []
    for name in LAUNCHES:
        monkeypatch.setattr(lib, name, lambda *a, name=name, launch=getattr(lib, name): (taken.append(name), launch(*a))[1])
    tokens = torch.randint(0, 256, (rows,), generator=torch.Generator().manual_seed(8)).tolist()

    def step():
        runner = ModelRunner(model, parsed, num_blocks=40, block_size=16, max_concurrent=9)
        if rows > 9:
            return runner.step([StepEntry(0, tokens, [rows - 1])]).clone()
        for i in range(rows):
            runner.step([StepEntry(i, (tokens * 20)[:20], [])])
        taken.clear()
        return runner.step([StepEntry(i, tokens[i:i + 1], [0]) for i in range(rows)]).clone()

    logits = step()
    rotated = [name for name in taken if name in LAUNCHES[:3] + LAUNCHES[5:]]
    assert set(rotated) == {rotates} and len(rotated) in (2, 4), taken  # (a short step runs once before it is recorded)
    assert not steady or "mi_gemm_tiles_bf16" not in taken
    monkeypatch.setattr(ops, "qkv_rope_write_many_plan", lambda *a: None)
    monkeypatch.setattr(ops, "qkv_rope_write_f32_takes", lambda *a: False)
    apart = step()
    if dtype == torch.float32 or steady or rows > 320 or kernels.tiles_for(rows, 1024, 512, False):
        assert torch.equal(logits, apart)
    else:  # (one product a layer in another order of sums: a bfloat16 rounding, 2^-9, of q, k and v, carried through two layers)
        assert (logits - apart).norm() < 2.0 ** -6 * apart.norm()


@pytest.mark.parametrize("m", [1, 7, 15, 17, 33, 63, 65, 130])
@pytest.mark.parametrize("n, k", [(16, 32), (37, 96), (200, 288), (64, 2048), (520, 4128), (130, 31), (33, 260)])
def test_every_form_of_the_float32_product_gives_the_same_bits(m, n, k):
    """Tiles of every size, in whole lines, in pieces and value by value, with rows and features beside whole tiles: the same order of the same
    64-bit sums; and against float64, which they round once (2^-24)."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import library
    from mini_infer_amd.ops.kernels import _ptr, _stream

    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    wide = torch.randn(n, (k + 31) // 32 * 32 + 32, generator=g, device="cuda")
    lib = library.load()
    a = torch.randn(m, k, generator=g, device="cuda")
    for first in (0, 4, 1):  # rows of W on a line, on 16 bytes, on neither
        w = wide[:, first : first + k]
        want = a.double() @ w.double().t()
        exact = want.float()
        got = ops.gemm_f32(a, w)
        assert ((got - exact).abs() <= 2.0 ** -23 * exact.abs() + 1e-12).all()
        for form in (0, 1, 2, 3, 4, 5, 7, 8):
            out = torch.full((m, n + 2), 7.0, device="cuda")
            library.check(lib.mi_gemm_f32_as(form, _ptr(a), a.stride(0), _ptr(w), w.stride(0), _ptr(out), out.stride(0), m, n, k, _stream()))
            assert torch.equal(out[:, :n], got) and (out[:, n:] == 7).all(), (first, form)


@pytest.mark.parametrize("m, n, k, first", [(13, 512, 160, 0), (43, 4096, 224, 0), (2, 1024, 145, 1), (11, 82, 140, 4), (136, 2048, 2048, 1), (232, 6418, 1024, 1),
                                            (150, 8192, 908, 4), (504, 3072, 512, 0), (383, 4096, 512, 0), (25, 2048, 2048, 0), (256, 2048, 8192, 0), (509, 3072, 2048, 0)])
def test_the_form_of_a_float32_product_is_near_the_fastest(m, n, k, first):
    """A few slices of K and many, operands in whole lines, in pieces and value by value; recorded, so that the host's part is not in it."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import library
    from mini_infer_amd.ops.kernels import _ptr, _stream

    lib = library.load()
    wide = torch.randn(n, (k + 31) // 32 * 32 + 32, device="cuda")
    a, w, out = torch.randn(m, k, device="cuda"), wide[:, first : first + k], torch.empty(m, n, device="cuda")

    def micros(product):
        product()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                product()
        times = []
        for _ in range(6):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            graph.replay()
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end) * 50)
        return min(times)

    def in_form(form):
        library.check(lib.mi_gemm_f32_as(form, _ptr(a), a.stride(0), _ptr(w), w.stride(0), _ptr(out), n, m, n, k, _stream()))

    fastest = min(micros(lambda form=form: in_form(form)) for form in (0, 1, 2, 3, 4, 5, 7, 8))
    assert micros(lambda: ops.gemm_f32(a, w)) < 1.3 * fastest


@pytest.mark.parametrize("tokens", [1, 3, 5, 8, 9, 17, 40, 130])
@pytest.mark.parametrize("heads, k, n", [(1, 64, 256), (32, 64, 256), (5, 256, 64), (3, 10, 22), (40, 36, 12)])
def test_float32_products_of_all_heads_are_those_of_each(tokens, heads, k, n):
    from mini_infer_amd import ops

    g = torch.Generator(device="cuda").manual_seed(tokens + heads)
    x = torch.randn(tokens, heads, k + 8, generator=g, device="cuda")[:, :, :k]
    w = torch.randn(heads, n, k, generator=g, device="cuda")
    out = torch.zeros(tokens, heads, n + 4, device="cuda")
    ops.linear_per_head(x, w, out[:, :, :n])
    for h in range(heads):
        assert torch.equal(out[:, h, :n], ops.gemm_f32(x[:, h], w[h]))
    assert (out[:, :, n:] == 0).all()


@pytest.mark.parametrize("heads, kv_heads, head_dim, v_dim", [(8, 2, 64, 64), (6, 2, 128, 128), (20, 2, 22, 30), (16, 1, 288, 256)])
@pytest.mark.parametrize("context", [5, 64, 101, 700])
def test_float32_attention_a_head_a_block_gives_the_bits_of_four(heads, kv_heads, head_dim, v_dim, context):
    """A token by itself (a block for each head) as one of many (four heads a block), with groups of fewer than four heads and ones that are not whole fours; the
    keys in ranges and not."""
    from mini_infer_amd.ops import kernels

    page, many = 16, 512 // heads + 1
    pages = -(-context // page)
    k_pages = _rand(pages + 2, kv_heads, page, head_dim, seed=81)
    v_pages = _rand(pages + 2, kv_heads, page, v_dim, seed=82)
    table = torch.randperm(pages, generator=torch.Generator().manual_seed(83)).to(torch.int32).to(DEV)[None]
    q = _rand(many, heads * head_dim, seed=84)

    def attended(rows, splits):
        n = rows.shape[0]
        out = torch.empty(n, heads * v_dim, device=DEV)
        names = dict(q_heads=heads, kv_heads=kv_heads, head_dim=head_dim, v_head_dim=v_dim, scale=head_dim ** -0.5, window=None, max_seq_len=context,
                     v_transposed=False, slopes=None, sink_logit=None, out=out)
        own = kernels.attention_splits
        kernels.attention_splits = lambda *a: splits
        try:
            return kernels._paged_attention_general(rows, k_pages, v_pages, table, torch.zeros(n, dtype=torch.int32, device=DEV),
                                                    torch.full((n,), context - 1, dtype=torch.int32, device=DEV), **names)
        finally:
            kernels.attention_splits = own

    for splits in (1, 3):
        together = attended(q, splits)
        for row in (0, many - 1):
            assert torch.equal(attended(q[row : row + 1], splits)[0], together[row]), (splits, row)
        if splits == 1:
            keys, values = (x[table[0].long()].transpose(1, 2).reshape(pages * page, kv_heads, -1)[:context].double() for x in (k_pages, v_pages))
            scores = torch.einsum("hd,chd->hc", q[0].view(heads, head_dim).double(), keys.repeat_interleave(heads // kv_heads, 1)) * head_dim ** -0.5
            exact = torch.einsum("hc,chd->hd", scores.softmax(1), values.repeat_interleave(heads // kv_heads, 1)).flatten()
            # (weights and result rounded to float32 once each)
            assert (together[0].double() - exact).norm() < 3e-7 * exact.norm()


@pytest.mark.parametrize("head_dim, v_dim", [(288, 256), (200, 144), (256, 250), (130, 130), (96, 64)])
@pytest.mark.parametrize("contexts", [[1, 64, 65], [300, 7, 129, 256, 257], [700]])
@pytest.mark.parametrize("window", [None, 100])
def test_float32_attention_over_wide_value_rows(head_dim, v_dim, contexts, window):
    """Values of up to 256 dims inside rows of keys, one key head, as few tokens as decoding brings (four waves share a range) and ends of
    64s: against float64, of which float32 results are one rounding (and one of each range's part) away."""
    from mini_infer_amd import ops

    g = torch.Generator(device="cuda").manual_seed(head_dim + sum(contexts))
    page, heads, tokens = 16, 6, len(contexts)
    width = -(-max(contexts) // page)
    pages = torch.randn(tokens * width, 1, page, head_dim, generator=g, device="cuda")
    table = torch.randperm(tokens * width, generator=g, device="cuda").int().view(tokens, width)
    q = torch.randn(tokens, heads * head_dim, generator=g, device="cuda")
    of = torch.arange(tokens, dtype=torch.int32, device="cuda")
    positions = torch.tensor(contexts, dtype=torch.int32, device="cuda") - 1
    cu = torch.arange(tokens + 1, dtype=torch.int32, device="cuda")
    got = ops.paged_attention(q, pages, None, table, of, positions, cu, cu.tolist(), q_heads=heads, kv_heads=1, head_dim=head_dim, scale=0.11,
                              window=window, max_seq_len=max(contexts), v_head_dim=v_dim)
    for t, n in enumerate(contexts):
        keys = pages[table[t].long()].view(-1, head_dim)[max(0, n - window) if window else 0 : n].double()
        p = torch.softmax(q[t].double().view(heads, head_dim) @ keys.t() * 0.11, -1)
        want = p @ keys[:, :v_dim]
        assert (got[t].double().view(heads, v_dim) - want).abs().max() < 2.0 ** -21 * want.abs().max()
