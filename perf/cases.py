"""What is timed when this engine is measured: steps of `ModelRunner.step`, as a serving program makes them.

A case is one step of one model: `prompt` (new requests, each given its whole prompt, logits at each one's last
token), `decode` (requests in the middle of their generation, one token each) or `mixed` (the same beside one portion
of a new prompt, the scheduler's ordinary step).  Models are the layer sizes of this repository's benchmark with random
weights: Llama at the 1B, 3B and 8B sizes, whole, and three of the other designs, 12 layers at those widths, one of
each kind of layer the engine has: gated delta rule and latent attention (Zekonex), gated linear attention and
state-space layers beside chunked attention (Kemurax), routed experts (Kunudra).  Llama comes in both types that the
engine computes in.

A decode pass goes on where the last one stopped, as generation does; its tokens are given, not sampled, so that a
tie between two logits does not send two runs different ways.
"""

from __future__ import annotations

import math
import random

import torch

from mini_infer_amd import ModelRunner, StepEntry
from mini_infer_amd.models import architecture_for

PAGE = 16
ROOM = 2048  # tokens a decoding request may still grow by before it is replaced by a new one
LAYERS = 12  # of the designs that the benchmark runs at Llama's widths
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
DEVICE = "cuda:0"


# -- models ---------------------------------------------------------------------------------------------------------

#        layers, width, heads, key/value heads, head size, feed-forward, tied head, frequency factor
SIZES = {
    "1b": (16, 2048, 32, 8, 64, 8192, True, 32.0),
    "3b": (28, 3072, 24, 8, 128, 8192, True, 32.0),
    "8b": (32, 4096, 32, 8, 128, 14336, False, 8.0),
}
VOCAB = 128256


def llama(size: str) -> dict:
    layers, width, heads, kv_heads, dim, ff, tied, factor = SIZES[size]
    return {
        "architectures": ["LlamaForCausalLM"], "num_hidden_layers": layers, "hidden_size": width, "num_attention_heads": heads,
        "num_key_value_heads": kv_heads, "head_dim": dim, "intermediate_size": ff, "vocab_size": VOCAB, "rope_theta": 500000.0,
        "rope_scaling": {"rope_type": "llama3", "factor": factor, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                         "original_max_position_embeddings": 8192},
        "rms_norm_eps": 1e-5, "tie_word_embeddings": tied, "max_position_embeddings": 131072,
    }


def zekonex(size: str) -> dict:
    """Delta rule, latent attention, delta rule, attention with a sink, and so on; a clamped feed-forward beside each."""
    _, width, heads, kv_heads, dim, ff, _, _ = SIZES[size]
    mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
    delta = {"type": "delta", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim, "conv": 4}}
    latent = {"type": "latent_attention", "mlp": mlp,
              "mixer": {"heads": heads, "dim": dim, "rot_dim": dim // 2, "vdim": dim, "kv_rank": 4 * dim, "scale": (dim + dim // 2) ** -0.5,
                        "rot": {"base": 10000.0, "dims": dim // 2}}}
    attention = {"type": "attention", "mlp": mlp,
                 "mixer": {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "rot": {"base": 500000.0, "dims": dim // 2}}}
    return {"architecture": "Zekonex", "vocab": VOCAB, "width": width, "embedding": {"scale": width ** 0.5}, "norm": {"eps": 1e-6},
            "residual_mult": 0.5, "layers": [(delta, latent, delta, attention)[i % 4] for i in range(LAYERS)]}


def kemurax(size: str) -> dict:
    """Gated linear attention, then three layers of chunked attention beside a state-space layer, and so on."""
    _, width, heads, kv_heads, dim, ff, _, _ = SIZES[size]
    mlp = {"kind": "dense", "ff": ff}
    gla = {"type": "gla", "mlp": mlp, "mixer": {"heads": width // 256, "dim": 128, "vdim": 256, "tau": 16.0}}
    left = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "mask": {"size": 8192},
            "rot": {"base": 500000.0, "dims": dim, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    right = {"heads": width // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
    pair = {"type": "parallel", "mlp": mlp, "mixer": {"left": left, "right": right, "left_scale": 0.5, "right_scale": 0.5}}
    return {"architecture": "Kemurax", "vocab": VOCAB, "width": width, "streams": 4, "norm": {"eps": 1e-6},
            "layers": [gla if i % 4 == 0 else pair for i in range(LAYERS)]}


def kunudra(size: str) -> dict:
    """Latent attention, two layers of capped attention, latent attention, and so on, all in a window; 16 experts, 2 a token."""
    _, width, heads, kv_heads, dim, ff, _, _ = SIZES[size]
    window = {"size": 1024}
    dense = {"kind": "dense", "ff": ff}
    moe = {"kind": "moe", "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}, "router": {"experts": 16, "identity": 2, "top": 2, "scale": 2.5}}
    attention = {"type": "attention",
                 "mixer": {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "mask": window, "softcap": 30.0, "v_mix": True}}
    latent = {"type": "latent_attention",
              "mixer": {"heads": heads, "dim": dim, "rot_dim": dim // 2, "vdim": dim, "kv_rank": 4 * dim, "q_rank": 12 * dim, "mask": window,
                        "scale": (dim + dim // 2) ** -0.5, "rot": {"base": 10000.0, "dims": dim // 2}}}
    return {"architecture": "Kunudra", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-6}, "postln_alpha": 1.6,
            "embedding": {"bigram": {"buckets": 65521, "mul_prev": 8191, "mul_cur": 31}},
            "layers": [dict((latent, attention, attention, latent)[i % 4], mlp=dense if i == 0 else moe) for i in range(LAYERS)]}


MODELS = {"llama": llama, "zekonex": zekonex, "kemurax": kemurax, "kunudra": kunudra}


def make_model(case: dict):
    """(config.json keys, parsed configuration, model without weights)."""
    raw = MODELS[case["model"]](case["size"])
    arch = architecture_for(raw)
    parsed = arch.parse_config(raw)
    return raw, parsed, arch.make_model(parsed, DTYPES[case["dtype"]], DEVICE)


def weights(model, seed: int):
    """name -> tensor, from the seed alone.  Matrices N(0, 0.02), those that write to the stream divided by the root of
    their number; norm weights around 1; the constants of the recurrences as such layers are initialised: rates between
    1 and 16, steps between 0.001 and 0.1, convolution taps of the size that four of them keep a channel's scale."""
    specs = model.param_specs()
    place = {name: i for i, name in enumerate(sorted(specs))}
    generator = torch.Generator(device=DEVICE)
    writes = 2.0 * len(model.blocks)

    def get(name: str) -> torch.Tensor:
        spec = specs[name]
        generator.manual_seed(seed * 1_000_003 + place[name])
        if name.endswith("A_log"):
            value = torch.log(1.0 + 15.0 * torch.rand(spec.shape, generator=generator, device=DEVICE))
        elif name.endswith("dt_bias"):
            step = torch.exp(math.log(1e-3) + math.log(100.0) * torch.rand(spec.shape, generator=generator, device=DEVICE))
            value = torch.log(torch.expm1(step))
        else:
            value = torch.randn(spec.shape, generator=generator, device=DEVICE)
            if spec.init == "norm_weight":
                value = 1.0 + 0.1 * value
            elif spec.init == "identity":
                value = torch.eye(*spec.shape, device=DEVICE) + 0.1 * value
            else:
                value = value * (0.3 if name.endswith(".conv") else 0.02)
                if name.endswith((".o", ".down", "o_proj.weight", "down_proj.weight")):
                    value = value * writes ** -0.5
        return value.to(torch.float32 if spec.dtype == "float32" else model.dtype)

    return get


# -- cases ----------------------------------------------------------------------------------------------------------


def _case(model, size, dtype, step, requests, context=0, tokens=0, name=None) -> dict:
    """`context`: positions the longest decoding request holds (they are spread from a quarter of it up); `tokens`: of
    the new prompt or prompts, together."""
    case = {"model": model, "size": size, "dtype": dtype, "step": step, "requests": requests, "context": context, "tokens": tokens}
    return case if name is None else {"name": name, **case}


def listed() -> list[dict]:
    return [
        # one user's chat on the smallest model: the smallest step there is, and the most often made
        _case("llama", "1b", "bfloat16", "decode", 1, context=1040, name="decode_1b_b1"),
        # the benchmark's headline: batch 8 at 8B sizes past a 2,048-token prompt
        _case("llama", "8b", "bfloat16", "decode", 8, context=2100, name="decode_8b_b8"),
        # a busy server: two dozen requests of mixed lengths
        _case("llama", "3b", "bfloat16", "decode", 24, context=3072, name="decode_3b_b24"),
        # time to first token of a long prompt
        _case("llama", "8b", "bfloat16", "prompt", 1, tokens=2048, name="prompt_8b_2048"),
        # the scheduler's step with its default portion beside a full house: 15 tokens decoded, 256 of a prompt
        _case("llama", "3b", "bfloat16", "mixed", 15, context=1500, tokens=256, name="mixed_3b_15_256"),
        # the 32-bit engine, which checkpoints are verified with: generation and a prompt
        _case("llama", "1b", "float32", "decode", 3, context=600, name="decode_1b_f32_b3"),
        _case("llama", "1b", "float32", "prompt", 1, tokens=509, name="prompt_1b_f32_509"),
        # recurrent designs: a prompt, several ragged prompts, a full house
        _case("zekonex", "8b", "bfloat16", "prompt", 1, tokens=2048, name="zekonex_prompt_2048"),
        _case("zekonex", "3b", "bfloat16", "decode", 30, context=700, name="zekonex_decode_b30"),
        _case("kemurax", "3b", "bfloat16", "prompt", 3, tokens=1777, name="kemurax_prompt_3x"),
        # routed experts: generation streams the chosen experts, a prompt visits them all
        _case("kunudra", "8b", "bfloat16", "decode", 8, context=1100, name="kunudra_decode_b8"),
        _case("kunudra", "3b", "bfloat16", "prompt", 2, tokens=1501, name="kunudra_prompt_2x"),
    ]


def _log_uniform(rng: random.Random, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random) -> dict:
    model = rng.choice(["llama", "llama", "llama", "zekonex", "kemurax", "kunudra"])
    wide = rng.random() < 0.2  # 32-bit
    size = "1b" if wide else rng.choice(list(SIZES))
    step = rng.choice(["prompt", "decode", "mixed"])
    most_requests, most_context, most_tokens = (6, 600, 509) if wide else (40, 2100, 2048)
    requests = context = tokens = 0
    if step == "prompt":
        tokens = _log_uniform(rng, 24, most_tokens)
        requests = rng.randint(1, max(1, min(4, tokens // 16)))
    else:
        requests = _log_uniform(rng, 1, most_requests)
        context = _log_uniform(rng, 64, most_context)
        if step == "mixed":
            tokens = _log_uniform(rng, 16, most_tokens // 2)
    return _case(model, size, "float32" if wide else "bfloat16", step, requests, context, tokens)


def _lengths(case: dict) -> tuple[list[int], list[int]]:
    """(positions each decoding request holds, tokens of each new prompt)."""
    n = case["requests"]
    if case["step"] == "prompt":
        each = case["tokens"] // n
        skew = [(i - (n - 1) / 2) / max(n - 1, 1) for i in range(n)]  # ragged: from half to one and a half of the mean
        prompts = [max(1, round(each * (1 + s))) for s in skew]
        prompts[-1] += case["tokens"] - sum(prompts)
        return [], prompts
    low = max(1, case["context"] // 4)
    held = [case["context"] - (case["context"] - low) * i // max(n - 1, 1) for i in range(n)]
    return held, [case["tokens"]] if case["step"] == "mixed" else []


def _tokens(case: dict, seed: int) -> tuple[list[list[int]], list[list[int]]]:
    """(every decoding request's tokens, those it will be given included; every new prompt's)."""
    held, prompts = _lengths(case)
    generator = torch.Generator().manual_seed(seed * 31 + 7)
    ids = lambda n: torch.randint(0, VOCAB, (n,), generator=generator).tolist()  # noqa: E731
    return [ids(n + ROOM) for n in held], [ids(n) for n in prompts]


# -- what is timed --------------------------------------------------------------------------------------------------


class State:
    """A serving program's side: its runner, its requests' tokens, and how far each request has come."""

    def __init__(self, case: dict, seed: int) -> None:
        _, parsed, model = make_model(case)
        model.load_params(weights(model, seed))
        self.held, self.prompt_lengths = _lengths(case)
        self.live, prompts = _tokens(case, seed)
        pages = sum(-(-len(t) // PAGE) + 1 for t in self.live + prompts) + 8
        self.runner = ModelRunner(model, parsed, num_blocks=pages, block_size=PAGE, max_concurrent=len(self.live) + len(prompts))
        self.new = [StepEntry(("new", i), t, [len(t) - 1]) for i, t in enumerate(prompts)]
        self.done = 0
        if self.live:
            self.begin()

    def begin(self) -> None:
        """The decoding requests' prompts, in portions, and one step of theirs."""
        for i, length in enumerate(self.held):
            if self.runner.has_request(i):
                self.runner.free_request(i)
            self.runner.step([StepEntry(i, self.live[i][:length], [])])
        self.done = 0
        self.runner.step(self.next_tokens())

    def next_tokens(self) -> list[StepEntry]:
        at = self.done
        self.done += 1
        return [StepEntry(i, [tokens[length + at]], [0]) for i, (tokens, length) in enumerate(zip(self.live, self.held))]


def prepare(case: dict, seed: int) -> State:
    return State(case, seed)


def run(state: State) -> torch.Tensor:
    """One step's logits."""
    if state.live and state.done == ROOM:
        state.begin()
    logits = state.runner.step((state.next_tokens() if state.live else []) + state.new)
    for entry in state.new:
        state.runner.free_request(entry.request_id)
    return logits


# -- what a step cannot do without ----------------------------------------------------------------------------------


def _attention_of(case: dict, raw: dict) -> list[tuple[int, int, int | None]]:
    """Per attention layer: (cached values a position, multiply-adds a query and key, window)."""
    if case["model"] == "llama":
        _, _, heads, kv_heads, dim, _, _, _ = SIZES[case["size"]]
        return [(2 * kv_heads * dim, 2 * heads * dim, None)] * raw["num_hidden_layers"]
    out = []
    for layer in raw["layers"]:
        m = layer["mixer"].get("left", layer["mixer"])
        if "kv_rank" in m:
            out.append((m["kv_rank"] + m["rot_dim"], m["heads"] * (2 * m["kv_rank"] + m["rot_dim"]), m.get("mask", {}).get("size")))
        elif "scale" in m:
            out.append((m["kv_heads"] * (m["dim"] + m["vdim"]), m["heads"] * (m["dim"] + m["vdim"]), m.get("mask", {}).get("size")))
    return out


def _states_of(case: dict, raw: dict) -> int:
    """Values of recurrent state a request keeps."""
    total = 0
    for layer in raw.get("layers", []):
        m = layer["mixer"].get("right", layer["mixer"])
        if layer["type"] in ("delta", "gla"):
            total += m["heads"] * m["dim"] * m["vdim"]
        elif layer["type"] == "parallel":
            total += m["heads"] * m["state"] * m["vdim"]
    return total


def work(case: dict) -> dict:
    raw, _, model = make_model(case)
    element = 2 if case["dtype"] == "bfloat16" else 4
    held, prompts = _lengths(case)
    tokens, rows = len(held) + sum(prompts), len(held) + len(prompts)
    width = SIZES[case["size"]][1]
    specs = model.param_specs()
    matrices = {n: math.prod(s.shape) for n, s in specs.items() if len(s.shape) == 2 and n not in ("embed", "bigram", "model.embed_tokens.weight", "head", "lm_head.weight")}
    experts = sum(v for n, v in matrices.items() if ".mlp.e" in n)
    fixed = sum(matrices.values()) - experts
    read, used = 0.0, 0.0
    if experts:  # 2 of 16 + 2 outputs a token, the last two of which have no weights
        chosen = 2 * 16 / 18
        read = experts * (1 - (1 - chosen / 16) ** tokens)
        used = experts / 16 * chosen * tokens
    head = VOCAB * width
    seen_bytes = seen_flops = 0.0
    for values, products, window in _attention_of(case, raw):
        w = window or 1 << 30
        keys = [min(n + 1, w) for n in held]
        pairs = sum(keys) + sum(sum(min(i + 1, w) for i in range(n)) for n in prompts)
        seen_bytes += (sum(keys) + sum(prompts)) * values * element
        seen_flops += 2.0 * products * pairs
    state = _states_of(case, raw)
    return {
        "bytes": (fixed + read + head + tokens * width) * element + seen_bytes + 4.0 * state * (2 * len(held) + len(prompts)) + 4.0 * rows * VOCAB,
        "flops": 2.0 * tokens * fixed + 2.0 * used + 2.0 * rows * head + seen_flops + 6.0 * tokens * state,
    }


def tolerance(case: dict) -> dict:
    """Four times what the logits of the first step were seen to differ from the same model's in 64 bits (0.021, 0.033 and
    0.05 for Llama at its three sizes, 0.0043, 0.01, and 4e-7 in 32 bits).  Where experts are routed most rows are
    0.004 off, but a token whose last two choices are close goes to another expert by rounding alone, and then its row
    is 0.1 off (0.034 for a step in which one of eight did)."""
    if case["dtype"] == "float32":
        return {"rel": 2e-6}
    if case["model"] == "llama":
        return {"rel": {"1b": 0.08, "3b": 0.13, "8b": 0.2}[case["size"]]}
    return {"rel": {"zekonex": 0.017, "kemurax": 0.04, "kunudra": 0.15}[case["model"]]}


# -- the same in 64 bits --------------------------------------------------------------------------------------------

MOST_FLOPS = 4e14  # above this `exact` would take too long


class Exact:
    """The designs in float64: whole sequences, no cache.  Rows are [requests, tokens, ...], short sequences filled up
    behind their end, where nothing they want sees it.  Rotation angles are the models' float32 numbers."""

    def __init__(self, raw: dict, weight) -> None:
        self.raw, self.weight = raw, weight

    def w(self, name: str) -> torch.Tensor:
        return self.weight(name).double()

    def linear(self, x: torch.Tensor, name: str) -> torch.Tensor:
        return x @ self.w(name).T

    @staticmethod
    def unit(x: torch.Tensor, eps: float) -> torch.Tensor:
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)

    @staticmethod
    def rotate(x: torch.Tensor, frequencies: torch.Tensor, interleaved: bool) -> torch.Tensor:
        """x [B, T, heads, d]: its first 2 * len(frequencies) entries turned by position."""
        half = frequencies.numel()
        angle = torch.arange(x.shape[1], device=x.device, dtype=torch.float32)[:, None] * frequencies.to(x.device, torch.float32)
        c, s = torch.cos(angle.double())[:, None], torch.sin(angle.double())[:, None]
        out = x.clone()
        first, second = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if interleaved else (slice(0, half), slice(half, 2 * half))
        a, b = x[..., first], x[..., second]
        out[..., first], out[..., second] = a * c - b * s, b * c + a * s
        return out

    @staticmethod
    def frequencies(base: float, dims: int) -> torch.Tensor:
        return torch.tensor(base, dtype=torch.float64) ** (-torch.arange(0, dims, 2, dtype=torch.float64) / dims)

    @staticmethod
    def rescaled(table: torch.Tensor, factor: float, low: float, high: float, original: int) -> torch.Tensor:
        wave = 2 * math.pi / table
        scaled = torch.where(wave > original / low, table / factor, table)
        smooth = (original / wave - low) / (high - low)
        between = (1 - smooth) * scaled / factor + smooth * scaled
        return torch.where((wave >= original / high) & (wave <= original / low), between, scaled)

    @staticmethod
    def attend(q, k, v, scale, window=None, chunk=None, sink=None, cap=None, slopes=None) -> torch.Tensor:
        """Causal attention of q [B, T, H, d] over k, v [B, T, G, ..]; `sink` [H]: a score without a value."""
        B, T, H, _ = q.shape
        per = H // k.shape[2]
        out = q.new_empty(B, T, H, v.shape[-1])
        for b in range(B):
            keys = k[b].permute(1, 2, 0).contiguous().repeat_interleave(per, 0)  # [H, d, T]
            values = v[b].transpose(0, 1).contiguous().repeat_interleave(per, 0)  # [H, T, dv]
            for at in range(0, T, 512):
                end = min(T, at + 512)
                s = torch.matmul(q[b, at:end].transpose(0, 1).contiguous(), keys[:, :, :end].contiguous()) * scale
                if cap is not None:
                    s = cap * torch.tanh(s / cap)
                i, j = torch.arange(at, end, device=q.device)[:, None], torch.arange(end, device=q.device)[None]
                if slopes is not None:
                    s = s - slopes[:, None, None] * (i - j)
                hidden = j > i
                if window is not None:
                    hidden = hidden | (j <= i - window)
                if chunk is not None:
                    hidden = hidden | (j < i // chunk * chunk)
                s = s.masked_fill(hidden, float("-inf"))
                top = s.amax(-1, keepdim=True)
                if sink is not None:
                    top = torch.maximum(top, sink[:, None, None])
                e = torch.exp(s - top)
                total = e.sum(-1, keepdim=True)
                if sink is not None:
                    total = total + torch.exp(sink[:, None, None] - top)
                out[b, at:end] = torch.matmul(e / total, values[:, :end].contiguous()).transpose(0, 1)
        return out

    # -- mixers

    def heads(self, x: torch.Tensor, name: str, count: int) -> torch.Tensor:
        return self.linear(x, name).unflatten(-1, (count, -1))

    def latent(self, h, p: str, m: dict, eps: float) -> torch.Tensor:
        H, d, rank = m["heads"], m["dim"], m["kv_rank"]
        table = self.frequencies(m["rot"]["base"], m["rot"]["dims"])
        if "q_rank" in m:
            q = self.heads(self.unit(self.linear(h, p + "dq"), eps) * self.w(p + "dq.norm"), p + "uq", H)
        else:
            q = self.heads(h, p + "q", H)
        down = self.linear(h, p + "dkv")
        c = self.unit(down[..., :rank], eps) * self.w(p + "dkv.norm")
        shared = self.rotate(down[..., None, rank:], table, True)
        q = torch.cat([q[..., :d], self.rotate(q[..., d:], table, True)], -1)
        k = torch.cat([self.heads(c, p + "uk", H), shared.expand(*shared.shape[:2], H, -1)], -1)
        return self.attend(q, k, self.heads(c, p + "uv", H), m["scale"], window=m.get("mask", {}).get("size"),
                           sink=self.w(p + "sink") if "mask" in m else None)

    def convolve(self, x: torch.Tensor, taps: torch.Tensor) -> torch.Tensor:
        n = taps.shape[1]
        padded = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
        return sum(taps[:, j] * padded[:, j : j + x.shape[1]] for j in range(n))

    def delta(self, h, p: str, m: dict, eps: float) -> torch.Tensor:
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (torch.nn.functional.silu(self.convolve(self.linear(h, p + n), self.w(f"{p}{n}.conv"))) for n in "qkv")
        q, k = (x.unflatten(-1, (G, d)) for x in (q, k))
        q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        q, k = ((x * f).repeat_interleave(H // G, 2) for x, f in ((q, d ** -0.5), (k, 1.0)))
        v = v.unflatten(-1, (H, -1))
        write = torch.sigmoid(self.linear(h, p + "b"))
        decay = torch.exp(-torch.exp(self.w(p + "A_log")) * torch.nn.functional.softplus(self.linear(h, p + "a") + self.w(p + "dt_bias")))
        S = h.new_zeros(h.shape[0], H, d, v.shape[-1])
        out = torch.empty_like(v)
        for t in range(h.shape[1]):
            S = S * decay[:, t, :, None, None]
            u = write[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S).squeeze(2))
            S = S + k[:, t, :, :, None] * u[:, :, None]
            out[:, t] = (q[:, t, :, None] @ S).squeeze(2)
        out = self.unit(out, eps) * self.w(p + "norm") * torch.nn.functional.silu(self.heads(h, p + "g", H))
        return out

    def linear_attention(self, h, p: str, m: dict, eps: float) -> torch.Tensor:
        H = m["heads"]
        q, k, v = self.heads(h, p + "q", H) * m["dim"] ** -0.5, self.heads(h, p + "k", H), self.heads(h, p + "v", H)
        z = self.linear(self.linear(h, p + "a1"), p + "a2") + self.w(p + "a2.b")
        alpha = torch.sigmoid(z).pow(1.0 / m["tau"]).unflatten(-1, (H, -1))
        out = self.scan(alpha, k, v, q)
        return (self.unit(out, eps) * self.w(p + "norm")).flatten(2) * torch.nn.functional.silu(self.linear(h, p + "g"))

    @staticmethod
    def scan(decay, k, v, q) -> torch.Tensor:
        """S = decay * S + k v^T, read out by q, token by token; decay [B, T, H, d or 1]."""
        S = v.new_zeros(v.shape[0], v.shape[2], k.shape[-1], v.shape[-1])
        out = torch.empty_like(v)
        for t in range(v.shape[1]):
            S = decay[:, t, :, :, None] * S + k[:, t, :, :, None] * v[:, t, :, None]
            out[:, t] = (q[:, t, :, None] @ S).squeeze(2)
        return out

    def state_space(self, h, p: str, m: dict, eps: float) -> torch.Tensor:
        H, N = m["heads"], m["state"]
        inner = H * m["vdim"]
        z, xbc, dt = self.linear(h, p + "in").split([inner, inner + 2 * N, H], -1)
        xbc = torch.nn.functional.silu(self.convolve(xbc, self.w(p + "conv")) + self.w(p + "conv.b"))
        x, B, C = xbc.split([inner, N, N], -1)
        x = x.unflatten(-1, (H, -1))
        step = torch.nn.functional.softplus(dt + self.w(p + "dt_bias"))
        decay = torch.exp(-torch.exp(self.w(p + "A_log")) * step)[..., None]
        B, C = (y[:, :, None].expand(-1, -1, H, -1) for y in (B, C))
        y = self.scan(decay, B * step[..., None], x, C) + self.w(p + "D")[:, None] * x
        return self.linear(self.unit(y.flatten(2) * torch.nn.functional.silu(z), eps) * self.w(p + "norm"), p + "o")

    # -- feed-forwards

    def gated(self, h, p: str, activation) -> torch.Tensor:
        return self.linear(activation(self.linear(h, p + "gate")) * self.linear(h, p + "up"), p + "down")

    def routed(self, h, p: str, mlp: dict) -> torch.Tensor:
        router, rows = mlp["router"], h.flatten(0, 1)
        s = torch.softmax(self.linear(rows, p + "router"), -1)
        chosen = torch.topk(s + self.w(p + "correction"), router["top"], -1).indices
        share = s.gather(-1, chosen) * router["scale"]
        out = rows * (share * (chosen >= router["experts"])).sum(-1, keepdim=True)
        for e in range(router["experts"]):
            at, place = torch.nonzero(chosen == e, as_tuple=True)
            if at.numel():
                out[at] += share[at, place, None] * self.gated(rows[at], f"{p}e{e}.", torch.nn.functional.silu)
        out = out + torch.sigmoid(self.linear(rows, p + "shared.sg")) * self.gated(rows, p + "shared.", torch.nn.functional.silu)
        return out.view_as(h)

    # -- stacks: tokens [B, T] -> logits at `last` [B]

    def pick(self, x, last) -> torch.Tensor:
        return x[torch.arange(x.shape[0], device=x.device), last]

    def llama(self, ids, last) -> torch.Tensor:
        c = self.raw
        H, G, d, eps = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"]
        r = c["rope_scaling"]
        table = 1.0 / (c["rope_theta"] ** (torch.arange(0, d, 2, dtype=torch.float32) / d))  # a float32 constant of the design
        table = self.rescaled(table, r["factor"], r["low_freq_factor"], r["high_freq_factor"], r["original_max_position_embeddings"])
        embed = self.weight("model.embed_tokens.weight")
        x = embed[ids].double()
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.unit(x, eps) * self.w(p + "input_layernorm.weight")
            q, k, v = (self.heads(h, f"{p}self_attn.{n}_proj.weight", n_heads) for n, n_heads in (("q", H), ("k", G), ("v", G)))
            a = self.attend(self.rotate(q, table, False), self.rotate(k, table, False), v, d ** -0.5)
            x = x + self.linear(a.flatten(2), p + "self_attn.o_proj.weight")
            h = self.unit(x, eps) * self.w(p + "post_attention_layernorm.weight")
            g, u = (self.linear(h, f"{p}mlp.{n}_proj.weight") for n in ("gate", "up"))
            x = x + self.linear(torch.nn.functional.silu(g) * u, p + "mlp.down_proj.weight")
        x = self.unit(self.pick(x, last), eps) * self.w("model.norm.weight")
        return x @ (embed if c["tie_word_embeddings"] else self.weight("lm_head.weight")).double().T

    def zekonex(self, ids, last) -> torch.Tensor:
        c = self.raw
        eps = c["norm"]["eps"]
        x = self.weight("embed")[ids].double() * c["embedding"]["scale"]
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = self.unit(x, eps) * self.w(f"l{i}.norm1")
            if layer["type"] == "delta":
                y = self.delta(h, p, m, eps)
            elif layer["type"] == "latent_attention":
                y = self.latent(h, p, m, eps)
            else:
                table = self.frequencies(m["rot"]["base"], m["rot"]["dims"])
                q, k = (self.rotate(self.heads(h, p + n, m[count]), table, True) for n, count in (("q", "heads"), ("k", "kv_heads")))
                y = self.attend(q, k, self.heads(h, p + "v", m["kv_heads"]), m["scale"], sink=h.new_zeros(m["heads"]))
            y = self.linear(y.flatten(2), p + "o")
            p, limit = f"l{i}.mlp.", layer["mlp"]["limit"]
            g = (self.linear(h, p + "gate") + self.w(p + "gate.b")).clamp(max=limit)
            u = (self.linear(h, p + "up") + self.w(p + "up.b")).clamp(-limit, limit)
            y = y + self.linear(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down") + self.w(p + "down.b")
            x = x + c["residual_mult"] * y
        return (self.unit(self.pick(x, last), eps) * self.w("final.norm")) @ self.w("head").T

    def kemurax(self, ids, last) -> torch.Tensor:
        c = self.raw
        eps = c["norm"]["eps"]
        norm = lambda y, name: self.unit(y, eps) * (1.0 + self.w(name))  # noqa: E731
        embed = self.weight("embed")
        xs = norm(embed[ids].double(), "embed.norm").expand(c["streams"], -1, -1, -1)
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            for n in (1, 2):
                read, write, mix = (self.w(f"l{i}.hc{n}.{k}") for k in ("in", "out", "mix"))
                h = norm(torch.tensordot(read, xs, 1), f"l{i}.norm{n}")
                if n == 2:
                    y = self.gated(h, f"l{i}.mlp.", lambda g: torch.nn.functional.gelu(g, approximate="tanh"))
                elif layer["type"] == "gla":
                    y = self.linear(self.linear_attention(h, p, m, eps), p + "o")
                else:
                    left, q = m["left"], p + "left."
                    s = left["rot"]["scaling"]
                    table = self.rescaled(self.frequencies(left["rot"]["base"], left["rot"]["dims"]), s["factor"], s["low"], s["high"], s["original"])
                    a, b = (self.rotate(self.unit(self.heads(h, q + k, left[count]), eps) * self.w(f"{q}{k}.norm"), table, False)
                            for k, count in (("q", "heads"), ("k", "kv_heads")))
                    y = self.attend(a, b, self.heads(h, q + "v", left["kv_heads"]), left["scale"], chunk=left["mask"]["size"])
                    y = self.linear(y.flatten(2) * torch.sigmoid(self.linear(h, q + "g")), q + "o")
                    y = m["left_scale"] * y + m["right_scale"] * self.state_space(h, p + "right.", m["right"], eps)
                xs = torch.tensordot(mix.T, xs, 1) + write[:, None, None, None] * y
        return norm(self.pick(xs.sum(0), last), "final.norm") @ embed.double().T

    def kunudra(self, ids, last) -> torch.Tensor:
        c = self.raw
        eps, alpha, pair = c["norm"]["eps"], c["postln_alpha"], c["embedding"]["bigram"]
        embed = self.weight("embed")
        row = torch.nn.functional.pad((ids[:, :-1] * pair["mul_prev"] + ids[:, 1:] * pair["mul_cur"]) % pair["buckets"], (1, 0), value=pair["buckets"])
        x = embed[ids].double() + self.weight("bigram")[row].double()
        v_first = None
        for i, layer in enumerate(c["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "latent_attention":
                y = self.latent(x, p, m, eps)
            else:
                q, k = (self.unit(self.linear(x, p + n), eps) * self.w(f"{p}{n}.norm") for n in "qk")
                v = self.linear(x, p + "v")
                if v_first is None:
                    v_first = v
                else:
                    v = torch.lerp(v, v_first, self.w(p + "vmix"))
                slopes = torch.pow(2.0, -8.0 * torch.arange(1, m["heads"] + 1, device=x.device, dtype=torch.float64) / m["heads"])
                y = self.attend(q.unflatten(-1, (m["heads"], -1)), k.unflatten(-1, (m["kv_heads"], -1)), v.unflatten(-1, (m["kv_heads"], -1)),
                                m["scale"], window=m["mask"]["size"], sink=self.w(p + "sink"), cap=m["softcap"], slopes=slopes)
            x = self.unit(alpha * x + self.w(f"l{i}.ls1") * self.linear(y.flatten(2), p + "o"), eps) * (1.0 + self.w(f"l{i}.norm1"))
            p = f"l{i}.mlp."
            y = self.gated(x, p, torch.nn.functional.silu) if layer["mlp"]["kind"] == "dense" else self.routed(x, p, layer["mlp"])
            x = self.unit(alpha * x + self.w(f"l{i}.ls2") * y, eps) * (1.0 + self.w(f"l{i}.norm2"))
        return (self.unit(self.pick(x, last), eps) * (1.0 + self.w("final.norm"))) @ embed.double().T


@torch.no_grad()
def exact(case: dict, seed: int) -> torch.Tensor | None:
    """The logits of a new state's first step, in 64 bits."""
    raw, _, model = make_model(case)
    held, prompts = _lengths(case)
    live, new = _tokens(case, seed)
    sequences = [tokens[: n + 2] for tokens, n in zip(live, held)] + new  # (a state's first step is its requests' second)
    matrix = sum(math.prod(s.shape) for n, s in model.param_specs().items() if len(s.shape) == 2 and n != "bigram" and ".mlp.e" not in n)
    if 2.0 * matrix * sum(len(s) for s in sequences) > MOST_FLOPS:
        return None
    stack = getattr(Exact(raw, weights(model, seed)), case["model"])
    rows: list[torch.Tensor | None] = [None] * len(sequences)
    order = sorted(range(len(sequences)), key=lambda i: -len(sequences[i]))
    while order:  # as many sequences at a time as make 16k tokens
        group = order[: max(1, 16384 // len(sequences[order[0]]))]
        order = order[len(group):]
        ids = torch.zeros(len(group), len(sequences[group[0]]), dtype=torch.int64)
        for at, i in enumerate(group):
            ids[at, : len(sequences[i])] = torch.tensor(sequences[i])
        last = torch.tensor([len(sequences[i]) - 1 for i in group], device=DEVICE)
        for i, row in zip(group, stack(ids.to(DEVICE), last)):
            rows[i] = row
    return torch.stack(rows)
