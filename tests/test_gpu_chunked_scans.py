"""The recurrences with a matrix state taken 32 tokens at a time, against the recurrence itself in 64 bits and
against the kernels that walk token by token."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = [([32, 31, 33, 1], 4, 2, 64, 64), ([200], 2, 2, 128, 128), ([97, 64, 5], 6, 3, 96, 80), ([129], 2, 1, 256, 250), ([65, 100], 3, 3, 20, 30),
         ([0, 70, 0, 33, 0], 18, 2, 64, 40)]  # (requests without tokens; more heads that share keys than a block takes at once)


def _rel(got, exact):
    return float((got.double() - exact).norm() / exact.norm())


def _state(generator, requests, shape, dim):
    state = torch.zeros(requests + 2, *shape, device=DEV)
    state[..., :dim] = torch.randn(requests + 2, *shape[:-1], dim, generator=generator, device=DEV) * 0.3
    return state


def _boundaries(lengths):
    return torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device=DEV)


def _rows(generator, tokens, width, odd):
    """bfloat16 rows; `odd`: of a buffer whose rows do not lie on 16 bytes."""
    wide = torch.randn(tokens, width + (3 if odd else 0), generator=generator, device=DEV).bfloat16()
    return wide[:, 3:] if odd else wide


def _calls_in_chunks(monkeypatch):
    """A list that grows by one with every call of the chunks' entry points."""
    from mini_infer_amd.ops import library

    lib, calls = library.load(), []
    for name in ("mi_gated_delta_chunks", "mi_decay_scan_chunks"):
        entry = getattr(lib, name)
        monkeypatch.setattr(lib, name, lambda *args, entry=entry: (calls.append(1), entry(*args))[1])
    return calls


def _both(monkeypatch, call, state):
    """What `call(state)` gives in chunks and token by token, with the state each leaves."""
    from mini_infer_amd.ops import kernels

    made, calls = [], _calls_in_chunks(monkeypatch)
    for chunks in (True, False):
        monkeypatch.setattr(kernels, "chunked_scan_pays", lambda walked, chunked, widest, chunks=chunks: chunks)
        left = state.clone()
        made.append((call(left), left))
        assert len(calls) == 1  # (the first call in chunks indeed, the second not)
    return made


def _check(chunked, walked, state, exact_out, exact_state, requests, dim, out_floor):
    (out, left), (out_walked, left_walked) = chunked, walked
    # float32 sums of up to 256 products and 32 tokens between two roundings of the state: a few 1e-7; never twice as far as
    # the kernel that rounds the state at every token
    assert _rel(left[:requests], exact_state) < max(4e-7, 2 * _rel(left_walked[:requests], exact_state))
    assert torch.equal(left[requests:], state[requests:])  # rows of other slots are not touched
    assert (left[..., dim:] == 0).all()
    assert _rel(out, exact_out) < max(out_floor, 2 * _rel(out_walked, exact_out))


def _exact_delta(qkv, proj, a_log, dt_bias, state, cu, heads, kv_heads, dim, vdim):
    """Normed and gated read-outs (norm weight 1) and the states left, in 64 bits."""
    tokens = qkv.shape[0]
    q, k, v = qkv.double().split([kv_heads * dim, kv_heads * dim, heads * vdim], 1)
    q, k = (x.view(tokens, kv_heads, dim) for x in (q, k))
    q, k = ((x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(heads // kv_heads, 1) for x in (q, k))
    v, p = v.view(tokens, heads, vdim), proj.double()
    write = torch.sigmoid(p[:, :heads])
    decay = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(p[:, heads : 2 * heads] + dt_bias.double()))
    out, left = torch.empty(tokens, heads, vdim, dtype=torch.float64, device=DEV), []
    for b in range(cu.numel() - 1):
        S = state[b].double()[..., :dim].transpose(1, 2)
        for t in range(int(cu[b]), int(cu[b + 1])):
            S = S * decay[t, :, None, None]
            S = S + k[t, :, :, None] * (write[t, :, None] * (v[t] - (k[t, :, None] @ S).squeeze(1)))[:, None]
            out[t] = (q[t, :, None] @ S).squeeze(1) * dim ** -0.5
        left.append(torch.nn.functional.pad(S.transpose(1, 2), (0, state.shape[-1] - dim)))
    out = out / torch.sqrt((out * out).mean(-1, keepdim=True) + 1e-6) * torch.nn.functional.silu(p[:, 2 * heads :].view(tokens, heads, vdim))
    return out.flatten(1), torch.stack(left)


@pytest.mark.parametrize("lengths,heads,kv_heads,dim,vdim", SIZES)
@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("fast", [False, True])
def test_gated_delta_in_chunks(monkeypatch, lengths, heads, kv_heads, dim, vdim, odd, fast):
    from mini_infer_amd import ops

    g = torch.Generator(device=DEV).manual_seed(7)
    tokens, requests = sum(lengths), len(lengths)
    qkv, proj = _rows(g, tokens, 2 * kv_heads * dim + heads * vdim, odd), _rows(g, tokens, 2 * heads + heads * vdim, odd)
    a_log = torch.log(1 + 15 * torch.rand(heads, generator=g, device=DEV))
    dt_bias = torch.full((heads,), 1.0 if fast else -4.0, device=DEV)  # fast: a state is forgotten within a few tokens
    weight = torch.ones(vdim, device=DEV)
    state = _state(g, requests, ops.delta_state_shape(heads, dim, vdim), dim)
    cu, slots = _boundaries(lengths), torch.arange(requests, dtype=torch.int32, device=DEV)
    chunked, walked = _both(monkeypatch, lambda s: ops.gated_delta(
        qkv, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, s, cu, slots, heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, eps=1e-6), state)

    out, left = _exact_delta(qkv, proj, a_log, dt_bias, state, cu, heads, kv_heads, dim, vdim)
    _check(chunked, walked, state, out, left, requests, dim, 2.0 ** -8)


@pytest.mark.parametrize("lengths", [[1], [1, 1, 1], [1, 0, 3, 0, 0], [0, 2]])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 2, 64, 64), (6, 3, 96, 80), (2, 1, 256, 250), (3, 3, 20, 30), (2, 2, 128, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gated_delta_of_decoded_tokens(lengths, heads, kv_heads, dim, vdim, dtype):
    """No more tokens than requests: one launch, whichever request the tokens belong to."""
    from mini_infer_amd import ops

    g = torch.Generator(device=DEV).manual_seed(11)
    tokens, requests = sum(lengths), len(lengths)
    qkv, proj = (_rows(g, tokens, n, True).to(dtype) for n in (2 * kv_heads * dim + heads * vdim, 2 * heads + heads * vdim))
    a_log, dt_bias = torch.rand(heads, generator=g, device=DEV), torch.full((heads,), -2.0, device=DEV)
    weight = 1 + 0.1 * torch.randn(vdim, generator=g, device=DEV)
    before = _state(g, requests, ops.delta_state_shape(heads, dim, vdim), dim)
    state = before.clone()
    cu, slots = _boundaries(lengths), torch.arange(requests, dtype=torch.int32, device=DEV)
    got = ops.gated_delta(qkv, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, state, cu, slots, heads=heads, kv_heads=kv_heads, dim=dim,
                          vdim=vdim, eps=1e-6)
    out, left = _exact_delta(qkv, proj, a_log, dt_bias, before, cu, heads, kv_heads, dim, vdim)
    # float32 state: a few roundings a token; what is written is rounded to the element type once
    assert _rel(state[:requests], left) < 2e-7 and torch.equal(state[requests:], before[requests:])
    assert _rel(got, out * weight.double().repeat(heads)) < (2.0 ** -8 if dtype == torch.bfloat16 else 3e-7)


@pytest.mark.parametrize("lengths,heads,groups,dim,vdim", SIZES)
@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("per_head", [False, True])
@pytest.mark.parametrize("fast", [False, True])
def test_decaying_state_in_chunks(monkeypatch, lengths, heads, groups, dim, vdim, odd, per_head, fast):
    from mini_infer_amd import ops

    if dim <= 32:
        dim = 40  # (narrower keys stay with the token-by-token kernel)
    g = torch.Generator(device=DEV).manual_seed(9)
    tokens, requests = sum(lengths), len(lengths)
    q, k, v = (_rows(g, tokens, n, odd) for n in (groups * dim, groups * dim, heads * vdim))
    gate = _rows(g, tokens, heads if per_head else heads * dim, odd) * (20.0 if fast else 1.0)
    bias = torch.full((heads if per_head else heads * dim,), -3.0 if per_head else 0.1, device=DEV)
    rate = torch.log(1 + 15 * torch.rand(heads, generator=g, device=DEV)) if per_head else None
    skip = torch.randn(heads, generator=g, device=DEV) if per_head else None
    state = _state(g, requests, ops.decay_state_shape(heads, dim, vdim), dim)
    cu, slots = _boundaries(lengths), torch.arange(requests, dtype=torch.int32, device=DEV)
    chunked, walked = _both(monkeypatch, lambda s: ops.decay_scan(
        q, 0, k, 0, v, 0, gate, 0, bias, s, cu, slots, heads=heads, groups=groups, dim=dim, vdim=vdim, per_head=per_head, rate=rate, skip=skip,
        inv_tau=0.0625, q_scale=0.125), state)

    qd, kd = (x.double().view(tokens, groups, dim).repeat_interleave(heads // groups, 1) for x in (q, k))
    x, z = v.double().view(tokens, heads, vdim), gate.double() + bias.double()
    if per_head:
        step = torch.nn.functional.softplus(z)
        decay, u = torch.exp(-torch.exp(rate.double()) * step)[..., None], x * step[..., None]
    else:
        decay, u = torch.sigmoid(z).pow(0.0625).view(tokens, heads, dim), x
    out, left = torch.empty(tokens, heads, vdim, dtype=torch.float64, device=DEV), []
    for b in range(requests):
        S = state[b].double()[..., :dim].transpose(1, 2)
        for t in range(int(cu[b]), int(cu[b + 1])):
            S = decay[t, :, :, None] * S + kd[t, :, :, None] * u[t, :, None]
            out[t] = (qd[t, :, None] @ S).squeeze(1) * 0.125
        left.append(torch.nn.functional.pad(S.transpose(1, 2), (0, state.shape[-1] - dim)))
    if per_head:
        out = out + skip.double()[:, None] * x
    _check(chunked, walked, state, out.flatten(1), torch.stack(left), requests, dim, 4e-7)


def test_rows_too_far_apart_for_chunks_go_token_by_token():
    from mini_infer_amd import ops

    heads, kv_heads, dim, vdim, tokens = 2, 1, 64, 64, 70
    g = torch.Generator(device=DEV).manual_seed(5)
    qkv = torch.randn(tokens, 2 * kv_heads * dim + heads * vdim, generator=g, device=DEV).bfloat16()
    far = torch.empty(tokens, 2**24, dtype=torch.bfloat16, device=DEV)[:, : qkv.shape[1]]
    far.copy_(qkv)
    proj = torch.randn(tokens, 2 * heads + heads * vdim, generator=g, device=DEV).bfloat16()
    a_log, dt_bias, weight = torch.zeros(heads, device=DEV), torch.full((heads,), -2.0, device=DEV), torch.ones(vdim, device=DEV)
    before = _state(g, 1, ops.delta_state_shape(heads, dim, vdim), dim)
    cu, slots = _boundaries([tokens]), torch.zeros(1, dtype=torch.int32, device=DEV)
    out, left = _exact_delta(qkv, proj, a_log, dt_bias, before, cu, heads, kv_heads, dim, vdim)
    for rows in (qkv, far):
        state = before.clone()
        got = ops.gated_delta(rows, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, state, cu, slots, heads=heads, kv_heads=kv_heads,
                              dim=dim, vdim=vdim, eps=1e-6)
        # as in the tests above: float32 states; read-outs rounded to bfloat16 once
        assert _rel(state[:1], left) < 4e-7 and _rel(got, out) < 2.0 ** -8


@pytest.mark.parametrize("kind", ["delta", "per_head", "per_channel"])
def test_a_rest_of_more_values_than_32_bits_count(kind):
    """520 value rows 2^23 apart: 519 of them are past 2^32 values.  The same bits as of rows side by side."""
    from mini_infer_amd import ops

    heads, groups, dim, vdim, tokens = 2, 1, 64, 64, 520
    g = torch.Generator(device=DEV).manual_seed(13)
    q, k, v = (torch.randn(tokens, n, generator=g, device=DEV).bfloat16() for n in (groups * dim, groups * dim, heads * vdim))
    rows = torch.cat([q, k, v], 1) if kind == "delta" else v
    far = torch.empty(tokens, 2**23, dtype=torch.bfloat16, device=DEV)[:, : rows.shape[1]]
    far.copy_(rows)
    cu, slots = _boundaries([tokens]), torch.zeros(1, dtype=torch.int32, device=DEV)
    made = []
    if kind == "delta":
        proj = torch.randn(tokens, 2 * heads + heads * vdim, generator=g, device=DEV).bfloat16()
        a_log, dt_bias, weight = torch.zeros(heads, device=DEV), torch.full((heads,), -2.0, device=DEV), torch.ones(vdim, device=DEV)
        before = _state(g, 1, ops.delta_state_shape(heads, dim, vdim), dim)
        for x in (rows, far):
            state = before.clone()
            made.append((ops.gated_delta(x, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, state, cu, slots, heads=heads,
                                         kv_heads=groups, dim=dim, vdim=vdim, eps=1e-6), state))
    else:
        per_head = kind == "per_head"
        gates = heads if per_head else heads * dim
        gate, bias = torch.randn(tokens, gates, generator=g, device=DEV).bfloat16(), torch.zeros(gates, device=DEV)
        before = _state(g, 1, ops.decay_state_shape(heads, dim, vdim), dim)
        for x in (rows, far):
            state = before.clone()
            made.append((ops.decay_scan(q, 0, k, 0, x, 0, gate, 0, bias, state, cu, slots, heads=heads, groups=groups, dim=dim, vdim=vdim,
                                        per_head=per_head, rate=torch.zeros(heads, device=DEV) if per_head else None, inv_tau=0.0625), state))
    assert torch.equal(made[0][0], made[1][0]) and torch.equal(made[0][1], made[1][1])


@pytest.mark.parametrize("dim,vdim", [(40, 64), (128, 128), (256, 250)])
@pytest.mark.parametrize("what", ["value inf", "value nan", "k inf", "q inf", "state inf", "state inf forgotten", "gate inf", "gate -inf", "gate nan"])
@pytest.mark.parametrize("kind", ["delta", "per_head", "per_channel"])
def test_what_is_not_finite_goes_token_by_token(monkeypatch, kind, what, dim, vdim):
    """A value, key, query, state or gate in the middle of a chunk that is no finite number reaches what it reaches in the
    token-by-token kernels: earlier tokens, other heads, other columns and other requests keep their numbers."""
    from mini_infer_amd import ops

    heads, groups, lengths, at, column = 4, 2, [50, 70], 50 + 32 + 9, 21
    tokens, requests = sum(lengths), len(lengths)
    g = torch.Generator(device=DEV).manual_seed(17)
    q, k, v = (torch.randn(tokens, n, generator=g, device=DEV).bfloat16() for n in (groups * dim, groups * dim, heads * vdim))
    per_channel = heads * dim if kind == "per_channel" else heads
    gate = torch.randn(tokens, per_channel, generator=g, device=DEV).bfloat16()
    shape = ops.delta_state_shape(heads, dim, vdim) if kind == "delta" else ops.decay_state_shape(heads, dim, vdim)
    state = _state(g, requests, shape, dim)
    name, bad, *forgotten = what.split()
    if forgotten:  # (a chunk's decays together are zero in float32, none of them by itself)
        gate[50:] = 40.0 if kind != "per_channel" else -100.0
    if name == "state":
        state[1, 1, column, 3] = float(bad)
    else:
        rows = {"value": (v, vdim + column), "k": (k, 7), "q": (q, 7), "gate": (gate, per_channel // heads)}[name]
        rows[0][at, rows[1]] = float(bad)
    cu, slots = _boundaries(lengths), torch.arange(requests, dtype=torch.int32, device=DEV)
    if kind == "delta":
        qkv = torch.cat([q, k, v], 1)
        proj = torch.cat([torch.randn(tokens, heads, generator=g, device=DEV).bfloat16(), gate, torch.randn(tokens, heads * vdim, generator=g, device=DEV).bfloat16()], 1)
        a_log, dt_bias, weight = torch.zeros(heads, device=DEV), torch.full((heads,), -2.0, device=DEV), torch.ones(vdim, device=DEV)
        call = lambda s: ops.gated_delta(qkv, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, s, cu, slots, heads=heads, kv_heads=groups, dim=dim, vdim=vdim, eps=1e-6)  # noqa: E731
    else:
        per_head = kind == "per_head"
        bias, rate = torch.zeros(per_channel, device=DEV), torch.zeros(heads, device=DEV) if per_head else None
        call = lambda s: ops.decay_scan(q, 0, k, 0, v, 0, gate, 0, bias, s, cu, slots, heads=heads, groups=groups, dim=dim, vdim=vdim, per_head=per_head, rate=rate, inv_tau=0.0625)  # noqa: E731
    (out, left), (out_walked, left_walked) = _both(monkeypatch, call, state)
    out, out_walked = out.double(), out_walked.double()
    for got, walked in ((out, out_walked), (left.double(), left_walked.double())):
        assert torch.equal(got.isnan(), walked.isnan()) and torch.equal(got.isinf(), walked.isinf()) and torch.equal(got[got.isinf()], walked[walked.isinf()])
        finite = walked.isfinite()
        # (bounds of the tests above: twice the error of one side against 64 bits)
        assert float((got - walked)[finite].norm() / walked[finite].norm()) < (2.0 ** -7 if kind == "delta" and got is out else 8e-7)
    assert out[: 50 if name == "state" else at].isfinite().all()


@pytest.mark.parametrize("heads,dim,vdim", [(16, 64, 64), (8, 256, 256)])
@pytest.mark.parametrize("kind", ["delta", "per_head", "per_channel"])
def test_what_is_not_finite_holds_a_step_up_no_longer_than_going_token_by_token(monkeypatch, kind, heads, dim, vdim):
    """A scan in chunks that takes its columns again, against the kernels that walk token by token alone: the chunks and the second walk together 1.1 to
    1.6 times their time (2.8 to 13 with each lane bringing its operands itself, and 1.7 with a decay per head of 64)."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    tokens, g = 1024, torch.Generator(device=DEV).manual_seed(29)
    q, k, v = (torch.randn(tokens, heads * n, generator=g, device=DEV).bfloat16() for n in (dim, dim, vdim))
    v[5] = float("nan")
    cu, slots = _boundaries([tokens]), torch.zeros(1, dtype=torch.int32, device=DEV)
    gates = heads * dim if kind == "per_channel" else heads
    gate, zeros = torch.randn(tokens, gates, generator=g, device=DEV).bfloat16(), torch.zeros(gates, device=DEV)
    state = _state(g, 1, ops.delta_state_shape(heads, dim, vdim) if kind == "delta" else ops.decay_state_shape(heads, dim, vdim), dim)
    qkv, proj = torch.cat([q, k, v], 1), torch.randn(tokens, 2 * heads + heads * vdim, generator=g, device=DEV).bfloat16()

    def scan():
        if kind == "delta":
            ops.gated_delta(qkv, proj, 0, heads, 2 * heads, zeros, zeros, torch.ones(vdim, device=DEV), state, cu, slots, heads=heads, kv_heads=heads, dim=dim,
                            vdim=vdim, eps=1e-6)
        else:
            ops.decay_scan(q, 0, k, 0, v, 0, gate, 0, zeros, state, cu, slots, heads=heads, groups=heads, dim=dim, vdim=vdim, per_head=kind == "per_head",
                           rate=zeros if kind == "per_head" else None, inv_tau=0.0625)

    took = []
    for chunks in (True, False):
        monkeypatch.setattr(kernels, "chunked_scan_pays", lambda *sizes, chunks=chunks: chunks)
        times = []
        for _ in range(6):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            scan()
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        took.append(min(times))
    assert took[0] < 2 * took[1], took


@pytest.mark.parametrize("lengths", [[1] * 5 + [40], [33, 1, 0, 1]])
@pytest.mark.parametrize("heads,shared,dim,vdim", [(4, 2, 64, 64), (2, 2, 128, 128), (6, 3, 96, 80), (2, 1, 256, 250), (4, 1, 40, 30), (18, 2, 64, 130)])
@pytest.mark.parametrize("kind", ["delta", "per_head", "per_channel"])
def test_single_tokens_beside_portions_in_chunks(monkeypatch, kind, lengths, heads, shared, dim, vdim):
    """Whole and partial groups of the column blocks that a single token's block takes together."""
    if kind == "delta":
        test_gated_delta_in_chunks(monkeypatch, lengths, heads, shared, dim, vdim, True, False)
    else:
        test_decaying_state_in_chunks(monkeypatch, lengths, heads, shared, dim, vdim, True, kind == "per_head", False)


@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 200)])
@pytest.mark.parametrize("kind", ["delta", "per_head", "per_channel"])
def test_single_tokens_that_are_not_finite(monkeypatch, kind, dim, vdim):
    """Beside a portion in chunks: as `test_what_is_not_finite_goes_token_by_token`, a request for each kind of it."""
    from mini_infer_amd import ops

    heads, groups, lengths, column = 4, 2, [1] * 8 + [40], vdim - 3
    tokens, requests = sum(lengths), len(lengths)
    g = torch.Generator(device=DEV).manual_seed(18)
    q, k, v = (torch.randn(tokens, n, generator=g, device=DEV).bfloat16() for n in (groups * dim, groups * dim, heads * vdim))
    per_channel = heads * dim if kind == "per_channel" else heads
    gate = torch.randn(tokens, per_channel, generator=g, device=DEV).bfloat16()
    state = _state(g, requests, ops.delta_state_shape(heads, dim, vdim) if kind == "delta" else ops.decay_state_shape(heads, dim, vdim), dim)
    v[0, vdim + column], v[1, column], k[2, 7], q[3, 7] = float("inf"), float("nan"), float("inf"), float("-inf")
    gate[4, 0], gate[5, 0], gate[6, 0], state[7, 1, column, 3] = float("inf"), float("-inf"), float("nan"), float("inf")
    cu, slots = _boundaries(lengths), torch.arange(requests, dtype=torch.int32, device=DEV)
    if kind == "delta":
        proj = torch.cat([torch.randn(tokens, heads, generator=g, device=DEV).bfloat16(), gate, torch.randn(tokens, heads * vdim, generator=g, device=DEV).bfloat16()], 1)
        names = dict(heads=heads, kv_heads=groups, dim=dim, vdim=vdim, eps=1e-6)
        made = _both(monkeypatch, lambda s: ops.gated_delta(torch.cat([q, k, v], 1), proj, 0, heads, 2 * heads, torch.zeros(heads, device=DEV),
                                                            torch.full((heads,), -2.0, device=DEV), torch.ones(vdim, device=DEV), s, cu, slots, **names), state)
    else:
        names = dict(heads=heads, groups=groups, dim=dim, vdim=vdim, per_head=kind == "per_head", inv_tau=0.0625,
                     rate=torch.zeros(heads, device=DEV) if kind == "per_head" else None)
        made = _both(monkeypatch, lambda s: ops.decay_scan(q, 0, k, 0, v, 0, gate, 0, torch.zeros(per_channel, device=DEV), s, cu, slots, **names), state)
    for got, walked in zip(*made):
        got, walked = got.double(), walked.double()
        assert torch.equal(got.isnan(), walked.isnan()) and torch.equal(got.isinf(), walked.isinf()) and torch.equal(got[got.isinf()], walked[walked.isinf()])
        finite = walked.isfinite()
        # (the read-out of the delta rule is rounded to bfloat16, else as above)
        assert float((got - walked)[finite].norm() / walked[finite].norm()) < (2.0 ** -7 if kind == "delta" and got.dim() == 2 else 8e-7)


# Requests in this order: single ones, portions and empty ones on both sides of the 64th from the end; more portions than a step of unknown division has blocks for.
MANY_REQUESTS = [[1] * 40 + [70], [1] * 10 + [33, 0] + [1] * 20 + [0, 0, 40] + [1] * 45 + [0, 65], [40, 33] * 32 + [1] * 20, [2] * 30 + [1] * 70 + [97]]


@pytest.mark.parametrize("lengths", MANY_REQUESTS)
@pytest.mark.parametrize("heads,shared,dim,vdim", [(16, 4, 64, 128), (18, 3, 96, 80), (6, 1, 256, 250)])
@pytest.mark.parametrize("known", [True, False])
@pytest.mark.parametrize("kind", ["delta", "per_channel"])
def test_chunks_of_steps_with_as_many_blocks_as_there_is_work(monkeypatch, kind, known, heads, shared, dim, vdim, lengths):
    """Where a walk's blocks find their pieces of work themselves (csrc/chunk_scan.h, launch_walk): every piece once, and those that a block makes one after
    another do not meet; a single token, a portion and a state that are not finite among them, and a request without a slot."""
    from mini_infer_amd import ops

    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    blocks, tokens, requests, longest = -(-vdim // 16), sum(lengths), len(lengths), max(lengths) if known else None
    assert requests * heads * blocks > 8 * cus and (kind != "delta" or heads * blocks < cus)
    portions = [b for b in range(requests) if lengths[b] > 1]
    many = 1 if longest is None else 1 + min(requests - 1, tokens - longest - (requests - 1))
    if many == requests:
        pytest.skip("a block for each request and its columns where the portions may be as many as the requests")
    if lengths is MANY_REQUESTS[2] and not known and dim != 96:
        assert heads * (len(portions) * blocks + 20 * 2) > 8 * cus  # (so blocks take a second piece)
    g = torch.Generator(device=DEV).manual_seed(31)
    q, k, v = (torch.randn(tokens, n, generator=g, device=DEV).bfloat16() for n in (shared * dim, shared * dim, heads * vdim))
    gate = torch.randn(tokens, heads * dim if kind == "per_channel" else heads, generator=g, device=DEV).bfloat16()
    state = _state(g, requests, ops.delta_state_shape(heads, dim, vdim) if kind == "delta" else ops.decay_state_shape(heads, dim, vdim), dim)
    cu = _boundaries(lengths)
    slots = torch.randperm(requests, generator=g, device=DEV).int()
    single, portion = lengths.index(1), portions[-1]
    slots[lengths.index(1, single + 1)] = -1
    v[int(cu[single]), vdim + 3], v[int(cu[portion]) + 1, vdim - 1] = float("nan"), float("inf")
    state[slots[lengths.index(1, single + 2)].long(), heads - 1, vdim - 1, 5] = float("inf")
    if kind == "delta":
        qkv = torch.cat([q, k, v], 1)
        proj = torch.cat([torch.randn(tokens, heads, generator=g, device=DEV).bfloat16(), gate, torch.randn(tokens, heads * vdim, generator=g, device=DEV).bfloat16()], 1)
        names = dict(heads=heads, kv_heads=shared, dim=dim, vdim=vdim, eps=1e-6, longest=longest)
        call = lambda s: ops.gated_delta(qkv, proj, 0, heads, 2 * heads, torch.zeros(heads, device=DEV), torch.full((heads,), -2.0, device=DEV),  # noqa: E731
                                         torch.ones(vdim, device=DEV), s, cu, slots, **names)
    else:
        names = dict(heads=heads, groups=shared, dim=dim, vdim=vdim, per_head=False, rate=None, inv_tau=0.0625, longest=longest)
        call = lambda s: ops.decay_scan(q, 0, k, 0, v, 0, gate, 0, torch.zeros(heads * dim, device=DEV), s, cu, slots, **names)  # noqa: E731
    (out, left), (out_walked, left_walked) = _both(monkeypatch, call, state)
    for got, walked in ((out.double(), out_walked.double()), (left.double(), left_walked.double())):
        assert torch.equal(got.isnan(), walked.isnan()) and torch.equal(got.isinf(), walked.isinf()) and torch.equal(got[got.isinf()], walked[walked.isinf()])
        finite = walked.isfinite()
        # (as test_what_is_not_finite_goes_token_by_token; a piece left out or made twice is some 1e-2)
        assert float((got - walked)[finite].norm() / walked[finite].norm()) < (2.0 ** -7 if kind == "delta" and got.dim() == 2 else 8e-7)
    assert torch.equal(left[requests:], state[requests:])


@pytest.mark.parametrize("kind", ["delta", "per_head", "per_channel"])
@pytest.mark.parametrize("lengths,known,chunks", [
    ([300], True, True), ([300], False, True), ([1] * 15 + [300], True, True), ([64] * 20, False, True),
    ([8] * 20, True, False), ([16] * 8, True, False), ([5] * 60, True, False), ([1] * 40, False, False), ([20] * 4, True, False), ([1] * 40, True, False),
])
def test_which_steps_go_in_chunks(monkeypatch, kind, lengths, known, chunks):
    """The rule by itself, on both sides of its line, with what the host knows of the portions and without."""
    from mini_infer_amd import ops

    calls = _calls_in_chunks(monkeypatch)
    heads, groups, dim, vdim, tokens = 16, 16, 128, 128, sum(lengths)
    cu, slots = _boundaries(lengths), torch.arange(len(lengths), dtype=torch.int32, device=DEV)
    rows = lambda n: torch.zeros(tokens, n, dtype=torch.bfloat16, device=DEV)  # noqa: E731
    longest = max(lengths) if known else None
    if kind == "delta":
        state = torch.zeros(len(lengths) + 1, *ops.delta_state_shape(heads, dim, vdim), device=DEV)
        per_head = torch.zeros(heads, device=DEV)
        ops.gated_delta(rows(2 * groups * dim + heads * vdim), rows(2 * heads + heads * vdim), 0, heads, 2 * heads, per_head, per_head,
                        torch.ones(vdim, device=DEV), state, cu, slots, heads=heads, kv_heads=groups, dim=dim, vdim=vdim, eps=1e-6, longest=longest)
    else:
        state = torch.zeros(len(lengths) + 1, *ops.decay_state_shape(heads, dim, vdim), device=DEV)
        gates = heads if kind == "per_head" else heads * dim
        ops.decay_scan(rows(groups * dim), 0, rows(groups * dim), 0, rows(heads * vdim), 0, rows(gates), 0, torch.zeros(gates, device=DEV), state,
                       cu, slots, heads=heads, groups=groups, dim=dim, vdim=vdim, per_head=kind == "per_head",
                       rate=torch.zeros(heads, device=DEV) if kind == "per_head" else None, longest=longest)
    assert len(calls) == int(chunks)


@pytest.mark.parametrize("lengths", [[1], [1, 0, 1, 1], [0, 3, 1, 0]])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(3, 3, 20, 30), (4, 2, 64, 250), (128, 4, 64, 40), (2, 1, 65, 16), (2, 2, 128, 128), (2, 1, 129, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gated_delta_of_steps_said_to_be_single_tokens(lengths, heads, kv_heads, dim, vdim, dtype):
    """On both sides of the key widths that the one launch takes; right also where a request brings more after all."""
    from mini_infer_amd import ops

    g = torch.Generator(device=DEV).manual_seed(19)
    tokens, requests = sum(lengths), len(lengths)
    qkv, proj = (_rows(g, tokens, n, True).to(dtype) for n in (2 * kv_heads * dim + heads * vdim, 2 * heads + heads * vdim))
    a_log, dt_bias, weight = torch.rand(heads, generator=g, device=DEV), torch.full((heads,), -2.0, device=DEV), torch.ones(vdim, device=DEV)
    before = _state(g, requests, ops.delta_state_shape(heads, dim, vdim), dim)
    state = before.clone()
    cu, slots = _boundaries(lengths), torch.arange(requests, dtype=torch.int32, device=DEV)
    got = ops.gated_delta(qkv, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, state, cu, slots, heads=heads, kv_heads=kv_heads, dim=dim,
                          vdim=vdim, eps=1e-6, longest=1)
    out, left = _exact_delta(qkv, proj, a_log, dt_bias, before, cu, heads, kv_heads, dim, vdim)
    # as for decoded tokens above
    assert _rel(state[:requests], left) < 2e-7 and torch.equal(state[requests:], before[requests:])
    assert _rel(got, out) < (2.0 ** -8 if dtype == torch.bfloat16 else 3e-7)


def test_a_recorded_step_is_not_taken_for_single_tokens():
    """No more tokens than requests, but one request's: the bits of the two launches, which steps of single tokens do not take."""
    from mini_infer_amd import ops

    heads, dim, tokens, requests = 4, 128, 8, 8
    g = torch.Generator(device=DEV).manual_seed(23)
    qkv, proj = (torch.randn(tokens, n, generator=g, device=DEV).bfloat16() for n in (3 * heads * dim, 2 * heads + heads * dim))
    a_log, dt_bias, weight = torch.zeros(heads, device=DEV), torch.full((heads,), -2.0, device=DEV), torch.ones(dim, device=DEV)
    before = _state(g, requests, ops.delta_state_shape(heads, dim, dim), dim)
    made = []
    for count in (requests, 1):  # (with one request there are more tokens than requests)
        state = before.clone()
        cu = torch.tensor([0] + [tokens] * count, dtype=torch.int32, device=DEV)
        made.append((ops.gated_delta(qkv, proj, 0, heads, 2 * heads, a_log, dt_bias, weight, state, cu, torch.arange(count, dtype=torch.int32, device=DEV),
                                     heads=heads, kv_heads=heads, dim=dim, vdim=dim, eps=1e-6), state))
    assert torch.equal(made[0][0], made[1][0]) and torch.equal(made[0][1], made[1][1])


@pytest.mark.parametrize("heads,groups,dim,vdim", [(4, 2, 64, 64), (6, 3, 96, 80), (2, 1, 256, 250), (3, 3, 20, 30), (2, 2, 128, 128), (2, 1, 12, 7), (300, 3, 40, 70),
                                                   (520, 2, 128, 20),
                                                   # four column blocks together: 4,096 blocks and more, a multiple of four a head
                                                   (300, 3, 40, 128), (300, 3, 20, 200), (270, 2, 128, 60), (258, 1, 256, 64), (130, 1, 12, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("odd", [False, True])
def test_decay_scan_of_single_tokens_gives_the_bits_of_portions(monkeypatch, heads, groups, dim, vdim, dtype, odd):
    """A decay per head: three tokens of a request in steps of one beside other portions, each with its state from memory, and as one portion
    (row runs read in pieces of 16 bytes and one by one); requests without tokens and one without a slot between them."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    monkeypatch.setattr(kernels, "chunked_scan_pays", lambda *sizes: False)
    g = torch.Generator(device=DEV).manual_seed(5)
    rows = [_rows(g, 3, 2 * groups * dim + heads * vdim + heads, odd).to(dtype) for _ in range(2)]  # of the two requests that are followed
    bias, rate, skip = (torch.randn(heads, generator=g, device=DEV) for _ in range(3))
    state = _state(g, 6, ops.decay_state_shape(heads, dim, vdim), dim)

    def step(parts, slots, into):
        x = torch.cat([p for p in parts if p is not None])
        if odd:
            x = torch.nn.functional.pad(x, (1, 0))[:, 1:]
        cu = _boundaries([0 if p is None else p.shape[0] for p in parts])
        return ops.decay_scan(x, 0, x, groups * dim, x, 2 * groups * dim, x, 2 * groups * dim + heads * vdim, bias, into, cu,
                              torch.tensor(slots, dtype=torch.int32, device=DEV), heads=heads, groups=groups, dim=dim, vdim=vdim, per_head=True,
                              rate=rate, skip=skip)

    whole, single = state.clone(), state.clone()
    out = step([rows[0], None, rows[1]], [3, 0, 1], whole)
    for t in range(3):
        portion = rows[0][:2] if t == 1 else None  # (steps of single tokens, and one with a portion)
        got = step([rows[0][t:t + 1], None, portion, rows[1][t:t + 1]], [3, 0, -1, 1], single)
        assert torch.equal(got[0], out[t]) and torch.equal(got[-1], out[3 + t])
    assert torch.equal(single[:-1], whole[:-1])


@pytest.mark.parametrize("heads,requests", [(65535, 257), (2, 65540)])
def test_decay_scan_of_more_blocks_than_a_launch_holds(heads, requests):
    """2^24 blocks and more, and more requests than a launch's third dimension takes: the same as in two steps."""
    from mini_infer_amd import ops

    dim, vdim = 12, 1
    g = torch.Generator(device=DEV).manual_seed(41)
    qk, v, gate = (torch.randn(requests, n, generator=g, device=DEV).bfloat16() for n in (2 * dim, heads * vdim, heads))
    bias, rate = torch.zeros(heads, device=DEV), torch.zeros(heads, device=DEV)
    state = _state(g, 1, ops.decay_state_shape(heads, dim, vdim), dim)
    slots = torch.full((requests,), -1, dtype=torch.int32, device=DEV)
    slots[0], slots[200] = 0, 1

    def scan(at, end, into):
        return ops.decay_scan(qk[at:end], 0, qk[at:end], dim, v[at:end], 0, gate[at:end], 0, bias, into, _boundaries([1] * (end - at)), slots[at:end].contiguous(),
                              heads=heads, groups=1, dim=dim, vdim=vdim, per_head=True, rate=rate)

    whole, parts = state.clone(), state.clone()
    out = scan(0, requests, whole)
    assert torch.equal(out, torch.cat([scan(0, 130, parts), scan(130, requests, parts)])) and torch.equal(whole, parts) and not torch.equal(whole, state)


def test_short_conv_of_more_rows_than_a_launch_holds():
    """2^27 + 9 rows of four channels: the last ones, which come behind 2^24 blocks of 8."""
    from mini_infer_amd import ops

    tokens, channels, g = 2**27 + 9, 4, torch.Generator(device=DEV).manual_seed(43)
    x = torch.zeros(tokens, channels, dtype=torch.bfloat16, device=DEV)
    x[-40:] = torch.randn(40, channels, generator=g, device=DEV).bfloat16()
    taps = torch.randn(channels, 4, generator=g, device=DEV)
    tail = torch.zeros(2, 3, channels, dtype=torch.bfloat16, device=DEV)
    cu, slots, of = _boundaries([tokens]), torch.zeros(1, dtype=torch.int32, device=DEV), torch.zeros(tokens, dtype=torch.int32, device=DEV)
    got = ops.short_conv(x, channels, taps, tail, cu, slots, of)
    last, own = x[-60:].contiguous(), torch.zeros(2, 3, channels, dtype=torch.bfloat16, device=DEV)
    want = ops.short_conv(last, channels, taps, own, _boundaries([60]), slots, of[:60].contiguous())
    assert torch.equal(got[-60:], want) and torch.equal(tail[0], own[0]) and not got[:-60].any()


def test_decay_scan_of_single_tokens_takes_few_heads_as_fast_as_many():
    """64 requests of 134 MB of states in 8 heads of 512 columns and in 64 of 64: 1.0 times (2.4 times where one block in four had work)."""
    from mini_infer_amd import ops

    dim, requests, g, took = 128, 64, torch.Generator(device=DEV).manual_seed(47), []
    cu, slots = _boundaries([1] * requests), torch.arange(requests, dtype=torch.int32, device=DEV)
    for heads, vdim in ((64, 64), (8, 512)):
        bias, rate = torch.zeros(heads, device=DEV), torch.zeros(heads, device=DEV)
        state = _state(g, requests, ops.decay_state_shape(heads, dim, vdim), dim)
        q, k, v, gate = (_rows(g, requests, n, False) for n in (dim, dim, heads * vdim, heads))
        times = []
        for _ in range(6):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            for _ in range(10):
                ops.decay_scan(q, 0, k, 0, v, 0, gate, 0, bias, state, cu, slots, heads=heads, groups=1, dim=dim, vdim=vdim, per_head=True, rate=rate)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        took.append(min(times))
    assert took[1] < 1.4 * took[0], took


def test_decay_scan_of_single_tokens_costs_little_more_off_16_bytes(monkeypatch):
    """Rows of q and k that cannot be read 16 bytes at a time: 1.1 times the time of those that can (1.5 times where every lane read its own value by value)."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    monkeypatch.setattr(kernels, "chunked_scan_pays", lambda *sizes: False)
    heads, dim, vdim, requests = 64, 256, 256, 8
    g = torch.Generator(device=DEV).manual_seed(37)
    bias, rate = torch.zeros(heads, device=DEV), torch.zeros(heads, device=DEV)
    state = _state(g, requests, ops.decay_state_shape(heads, dim, vdim), dim)
    cu, slots = _boundaries([1] * requests), torch.arange(requests, dtype=torch.int32, device=DEV)
    took = []
    for odd in (False, True):
        q, k, v, gate = (_rows(g, requests, n, odd) for n in (dim, dim, heads * vdim, heads))
        times = []
        for _ in range(6):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            for _ in range(10):
                ops.decay_scan(q, 0, k, 0, v, 0, gate, 0, bias, state, cu, slots, heads=heads, groups=1, dim=dim, vdim=vdim, per_head=True, rate=rate)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        took.append(min(times))
    assert took[1] < 1.3 * took[0], took


@pytest.mark.parametrize("lengths,channels", [([1, 2, 3, 0, 4, 1, 5, 9, 1], 12), ([70], 1028), ([3, 1] * 8 + [17, 6, 1, 2], 96),
                                              ([1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 300, 3], 8192), ([2, 1, 3, 990, 13, 4, 1, 1, 29], 8192)])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_short_conv_of_rows_in_fours_gives_the_bits_of_the_general_form(lengths, channels, taps, dtype):
    """One, four and eight rows a thread (by the step's size), requests that begin and end anywhere in them, twice in a row so that tails are carried:
    against rows off 16 bytes, which take the launches that stand for any layout."""
    from mini_infer_amd import ops

    g = torch.Generator(device=DEV).manual_seed(sum(lengths))
    requests, tokens = len(lengths), sum(lengths)
    w, bias = torch.randn(channels, taps, generator=g, device=DEV), torch.randn(channels, generator=g, device=DEV)
    slots = torch.randperm(requests, generator=g, device=DEV).int()
    of = torch.repeat_interleave(torch.arange(requests, device=DEV), torch.tensor(lengths, device=DEV)).int()
    tail = torch.randn(requests + 1, taps - 1, channels, generator=g, device=DEV).to(dtype)
    other = tail.clone()
    for _ in range(2):
        x = torch.randn(tokens, channels, generator=g, device=DEV).to(dtype)
        off = torch.empty(tokens, channels + 1, dtype=dtype, device=DEV)[:, :channels].copy_(x)
        assert torch.equal(ops.short_conv(x, channels, w, tail, _boundaries(lengths), slots, of, bias=bias),
                           ops.short_conv(off, channels, w, other, _boundaries(lengths), slots, of, bias=bias))
        assert torch.equal(tail, other)


@pytest.mark.parametrize("kind", ["decay", "channels", "delta"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("chunks", [False, True])
@pytest.mark.parametrize("lengths", [[1, 1, 1, 1], [1, 40, 2, 33]])
def test_requests_without_a_slot_start_from_the_spare_row_and_leave_it_as_it_is(monkeypatch, kind, dtype, chunks, lengths):
    """Rows that only fill a recorded step: what they would give with a slot that holds what the spare row does, while no row of the state is
    written for them."""
    from mini_infer_amd import ops
    from mini_infer_amd.ops import kernels

    if chunks and dtype == torch.float32:
        pytest.skip("chunks are of bfloat16 rows")
    monkeypatch.setattr(kernels, "chunked_scan_pays", lambda *sizes: chunks)
    heads, dim, vdim, tokens = 4, 128, 64, sum(lengths)
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(tokens, 4 * heads * (dim + vdim), generator=g, device=DEV).to(dtype)
    bias, rate = torch.randn(heads * dim, generator=g, device=DEV), torch.rand(heads, generator=g, device=DEV)
    shape = ops.delta_state_shape(heads, dim, vdim) if kind == "delta" else ops.decay_state_shape(heads, dim, vdim)
    state = torch.randn(6, *shape, generator=g, device=DEV)
    state[4] = state[5]
    cu = _boundaries(lengths)

    def step(slots, into):
        slots = torch.tensor(slots, dtype=torch.int32, device=DEV)
        if kind == "delta":
            return ops.gated_delta(x, x, 0, heads, 2 * heads, rate, bias[:heads], torch.ones(vdim, device=DEV), into, cu, slots, heads=heads, kv_heads=heads,
                                   dim=dim, vdim=vdim, eps=1e-6)
        per_head = kind == "decay"
        return ops.decay_scan(x, 0, x, heads * dim, x, 2 * heads * dim, x, 2 * heads * dim + heads * vdim, bias[: heads if per_head else heads * dim], into, cu,
                              slots, heads=heads, groups=heads, dim=dim, vdim=vdim, per_head=per_head, rate=rate if per_head else None)

    left, zeros = state.clone(), state.clone()
    got, want = step([2, -1, 0, -1], left), None
    rows = [torch.arange(int(cu[b]), int(cu[b + 1]), device=DEV) for b in range(4)]
    want = step([2, 4, 0, 3], zeros)
    assert torch.equal(got[rows[0]], want[rows[0]]) and torch.equal(got[rows[1]], want[rows[1]]) and torch.equal(got[rows[2]], want[rows[2]])
    assert torch.equal(left[[0, 2]], zeros[[0, 2]]) and torch.equal(left[[1, 3, 4, 5]], state[[1, 3, 4, 5]])
