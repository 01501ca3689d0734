"""The decode-path workloads whose speed this framework answers for.

Each case is one call (or one short sequence of calls) of the public torch
mirror `ppk` as a decode loop makes it, on synthetic data drawn on the GPU
from a seed. The history follows the benchmark's heavy-tail rule: N(0, 1),
except 2 % of the (head, channel) pairs, which hold 10 * Student-t(3).

Operations ("op"):
  decode   int8 KV cache: append of the current token + attention
           (ppk.DecodeStep), or attention alone (ppk.DecodeAttention), over
           `layers` independent layers
  float    the same over a bf16 / f32 KV store (ppk.FloatDecodeStep,
           ppk.FloatDecodeAttention)
  append   quantize-and-append of `tokens` new tokens per sequence
           (ppk.AppendKV) into `layers` layers' arenas
  codec    ppk.quantize of a dense tensor, then ppk.dequantize of its codes
  arena    one decode round of a KV cache manager: a shared write plan, then
           per layer a reserving batch write and the fused decode step
  sample   the CFG + Renyi sampler (ppk.RenyiSampler)
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "pop2-bezier_amd"))

import ppk  # noqa: E402
from ppk.kv_arena import LayerCache, WritePlan  # noqa: E402
from ppk.kv_arena import decode_step as arena_decode_step  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ELEM = {"f32": 4, "bf16": 2, "f16": 2}
DEVICE = "cuda:0"

# No drawn case moves more than the headline step does (one 8192-token int8 history
# of 512 head rows at D = 128).
MOST_BYTES = 1_110_000_000
MOST_STATE_BYTES = 3_000_000_000


def listed():
    return [
        # The smallest step: one sequence, 512 cached tokens, everything f32
        # (the reference's model width, D = 64). Launch- and latency-bound.
        _decode("decode_b1_512_d64", 1, 16, 64, 512, capacity=1024, q="f32"),
        # One token of one sequence through a 24-layer model, 2048 cached tokens.
        _decode("decode_24layers_b1_2048_d128", 1, 16, 128, 2048, capacity=2049, layers=24),
        # A serving batch of eight sequences of 256 to 4096 tokens, lengths
        # known on the host.
        _decode("decode_b8_ragged_4096_d128", 8, 16, 128, 4096, capacity=4097, least=256, host=True),
        # A mid-size serving batch in a power-of-two arena, bf16 output, lengths
        # on the device only.
        _decode("decode_b16_1500_d64", 16, 16, 64, 1500, capacity=2048, least=1200, out="bf16"),
        # The headline: 32 sequences of 8192 tokens.
        _decode("decode_b32_8192_d128", 32, 16, 128, 8192, capacity=8193),
        # The option that rounds every history element to bf16, as the
        # reference's own kernel does, at the reference's head width.
        _decode("decode_bf16_history_b32_4096_d64", 32, 16, 64, 4096, capacity=4097, bf16_history=True),
        # The graph-decode session: fused write + attention over a 1024-token
        # bf16 store, f32 queries.
        _float("float_step_b16_1024_d64", 16, 16, 64, 1000, capacity=1024, least=200, step=True),
        # Attention over a ragged bf16 store, lengths known on the host.
        _float("float_b32_ragged_8192_d128", 32, 16, 128, 8192, capacity=8192, least=256, host=True),
        # A prompt's K and V quantized into the int8 arenas.
        _append("append_prefill_b32_1000_d128", 32, 16, 128, 1000, capacity=2048, past=24),
        # A dense tensor to int8 and back (the transient prefix of a prefill).
        {"name": "codec_512x2048_d128", "op": "codec", "rows": 512, "tokens": 2048, "head_dim": 128, "src": "bf16",
         "out": "bf16"},
        # A decode round of a cache manager over 24 layers of 16 sequences.
        {"name": "arena_round_24x16_d64", "op": "arena", "layers": 24, "batch": 16, "heads": 16, "head_dim": 64,
         "tokens": 700, "least": 300, "lengths_seed": 5, "q": "bf16"},
        # The head of a guided decode step.
        {"name": "sample_b32_2048", "op": "sample", "batch": 32, "guidance": 2, "choices": 2048, "alpha": 4.0,
         "cfg": 2.5, "least_legal": 2048},
    ]


def _decode(name, batch, heads, head_dim, tokens, *, capacity, least=0, host=False, layers=1, q="bf16", out="f32",
            bf16_history=False, step=True, lengths_seed=1):
    return {"name": name, "op": "decode", "batch": batch, "heads": heads, "head_dim": head_dim, "tokens": tokens,
            "least": least or tokens, "lengths_seed": lengths_seed, "host": host, "capacity": capacity,
            "layers": layers, "q": q, "out": out, "bf16_history": bf16_history, "step": step}


def _float(name, batch, heads, head_dim, tokens, *, capacity, least=0, host=False, kv="bf16", q="f32", out="f32",
           step=False, lengths_seed=1):
    return {"name": name, "op": "float", "batch": batch, "heads": heads, "head_dim": head_dim, "tokens": tokens,
            "least": least or tokens, "lengths_seed": lengths_seed, "host": host, "capacity": capacity, "kv": kv,
            "q": q, "out": out, "step": step}


def _append(name, batch, heads, head_dim, tokens, *, capacity, past, layers=1, src="bf16"):
    return {"name": name, "op": "append", "batch": batch, "heads": heads, "head_dim": head_dim, "tokens": tokens,
            "past": past, "capacity": capacity, "layers": layers, "src": src}


def _spread(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    op = rng.choice(["decode", "decode", "decode", "float", "float", "append", "codec", "arena", "sample"])
    while True:
        case = _DRAW[op](rng)
        case["op"] = op
        case.pop("name", None)
        if work(case)["bytes"] <= MOST_BYTES and _state_bytes(case) <= MOST_STATE_BYTES:
            return case


def _draw_lengths(rng, tokens):
    """Uniform batches, or ragged ones down to a sixteenth of the longest."""
    return tokens if rng.random() < 0.5 else max(1, tokens // rng.randint(2, 16))


def _draw_capacity(rng, tokens):
    kind = rng.randrange(3)
    if kind == 0:
        return tokens + 1
    if kind == 1:
        return 1 << tokens.bit_length()
    return tokens + 1 + rng.randrange(1, 500)


def _draw_decode(rng):
    tokens = _spread(rng, 16, 16384)
    c = _decode("", _spread(rng, 1, 64), rng.choice([8, 16, 16, 32]), rng.choice([64, 64, 128, 128, 256]), tokens,
                capacity=_draw_capacity(rng, tokens), least=_draw_lengths(rng, tokens), host=rng.random() < 0.5,
                q=rng.choice(["bf16", "f32", "f16"]), out=rng.choice(["f32", "bf16"]),
                bf16_history=rng.random() < 0.2, step=rng.random() < 0.75, lengths_seed=rng.randrange(10**6))
    if rng.random() < 0.3:
        c["layers"] = rng.randint(2, 24)
    return c


def _draw_float(rng):
    tokens = _spread(rng, 16, 8192)
    return _float("", _spread(rng, 1, 64), rng.choice([8, 16, 16, 32]), rng.choice([64, 64, 128, 128, 256]), tokens,
                  capacity=_draw_capacity(rng, tokens), least=_draw_lengths(rng, tokens), host=rng.random() < 0.5,
                  kv=rng.choice(["bf16", "bf16", "f32"]), q=rng.choice(["f32", "bf16"]),
                  out=rng.choice(["f32", "bf16"]), step=rng.random() < 0.6, lengths_seed=rng.randrange(10**6))


def _draw_append(rng):
    tokens, past = _spread(rng, 1, 4000), rng.randrange(0, 2000)
    c = _append("", _spread(rng, 1, 64), rng.choice([8, 16, 32]), rng.choice([64, 128, 256]), tokens,
                capacity=_draw_capacity(rng, tokens + 2 * past), past=past, src=rng.choice(["bf16", "f16", "f32"]))
    if tokens < 16:
        c["layers"] = rng.randint(4, 24)
    return c


def _draw_codec(rng):
    return {"rows": _spread(rng, 16, 1024), "tokens": _spread(rng, 1, 8192), "head_dim": rng.choice([64, 128, 256]),
            "src": rng.choice(["bf16", "f16", "f32"]), "out": rng.choice(["bf16", "f32", "f16"])}


def _draw_arena(rng):
    tokens = _spread(rng, 32, 2000)
    return {"layers": rng.randint(4, 24), "batch": _spread(rng, 1, 32), "heads": rng.choice([8, 16]),
            "head_dim": rng.choice([64, 128]), "tokens": tokens, "least": _draw_lengths(rng, tokens),
            "lengths_seed": rng.randrange(10**6), "q": rng.choice(["bf16", "f32"])}


def _draw_sample(rng):
    choices, guidance = _spread(rng, 16, 2048), rng.choice([1, 2])
    return {"batch": _spread(rng, 1, 256), "guidance": guidance, "choices": choices,
            "alpha": rng.choice([2.0, 4.0, 6.5]), "cfg": 1.0 if guidance == 1 else rng.choice([1.5, 2.5, 4.0]),
            "least_legal": max(1, choices // rng.choice([1, 1, 4]))}


_DRAW = {"decode": _draw_decode, "float": _draw_float, "append": _draw_append, "codec": _draw_codec,
         "arena": _draw_arena, "sample": _draw_sample}


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
def lengths_of(case) -> list[int]:
    """The sequences' stored tokens: the longest holds case["tokens"], the others down to case["least"]."""
    rng = random.Random(case["lengths_seed"])
    got = [rng.randint(case["least"], case["tokens"]) for _ in range(case["batch"])]
    got[rng.randrange(case["batch"])] = case["tokens"]
    return got


def work(case) -> dict:
    op = case["op"]
    if op == "sample":
        values = case["batch"] * case["choices"]
        return {"bytes": values * case["guidance"] * 4 + case["batch"] * (12 + 12), "flops": 8 * values}
    d = case["head_dim"]
    if op == "codec":
        n = case["rows"] * case["tokens"]
        return {"bytes": n * d * (ELEM[case["src"]] + 1) + 4 * n + n * (d + 4) + n * d * ELEM[case["out"]],
                "flops": 4 * n * d}
    rows = case["batch"] * case["heads"]
    if op == "append":
        n = case["layers"] * 2 * rows * case["tokens"]
        return {"bytes": n * (d * ELEM[case["src"]] + d + 4), "flops": 3 * n * d}
    tokens = case["heads"] * sum(lengths_of(case))
    q = ELEM[case["q"]]
    if op == "float":
        e = ELEM[case["kv"]]
        new = rows * d * 2 * (q + e) if case["step"] else 0
        return {"bytes": tokens * 2 * d * e + rows * d * (q + ELEM[case["out"]]) + new,
                "flops": 4 * d * (tokens + rows)}
    out = ELEM[case.get("out", "f32")]
    new = rows * 2 * (d + 4) if case.get("step", True) else 0
    layer = tokens * 2 * (d + 4) + rows * d * (3 * q + out) + new  # q, current K and V read once each
    return {"bytes": case["layers"] * layer, "flops": case["layers"] * 4 * d * (tokens + rows)}


def _state_bytes(case) -> int:
    op = case["op"]
    if op in ("sample", "codec"):
        return work(case)["bytes"]
    rows, d = case["batch"] * case["heads"], case["head_dim"]
    if op == "float":
        return rows * case["capacity"] * 2 * d * ELEM[case["kv"]]
    if op == "arena":
        return case["layers"] * rows * 4 * case["tokens"] * 2 * (d + 4)
    return case["layers"] * rows * case["capacity"] * 2 * (d + 4) + (work(case)["bytes"] if op == "append" else 0)


# ---------------------------------------------------------------------------
# Inputs: plain torch, the same for prepare() and exact()
# ---------------------------------------------------------------------------
class _Draw:
    """Seeded tensors on the GPU, one generator per named tensor."""

    def __init__(self, seed: int):
        self.seed = seed

    def _gen(self, name: str) -> torch.Generator:
        h = 1469598103934665603
        for ch in f"{self.seed}/{name}":
            h = ((h ^ ord(ch)) * 1099511628211) % 2**61
        return torch.Generator(device=DEVICE).manual_seed(h)

    def normal(self, name, shape, dtype="f32"):
        return torch.randn(shape, generator=self._gen(name), device=DEVICE).to(DTYPES[dtype])

    def history(self, name, batch, heads, tokens, d):
        """f32 [batch * heads, tokens, d], 2 % of the (head, channel) pairs heavy-tailed."""
        g = self._gen(name)
        x = torch.randn((batch, heads, tokens, d), generator=g, device=DEVICE)
        pairs = torch.randperm(heads * d, generator=g, device=DEVICE)[:max(1, round(0.02 * heads * d))].sort().values
        for p in pairs.tolist():
            z = torch.randn((4, batch, tokens), generator=g, device=DEVICE)
            x[:, p // d, :, p % d] = 10.0 * z[0] / torch.sqrt(z[1:].square().sum(0) / 3.0)
        return x.reshape(batch * heads, tokens, d)


def _quantized(x):
    """The int8 rule on f32 [rows, tokens, d]: codes (two's complement bytes) and per-token scales."""
    codes = torch.empty(x.shape, dtype=torch.uint8, device=x.device)
    scales = torch.empty(x.shape[:2], dtype=torch.float32, device=x.device)
    top = torch.full((), 127.0, device=x.device)  # a tensor: torch divides by a plain number through its reciprocal
    for r in range(0, x.shape[0], 64):
        part = x[r:r + 64]
        s = torch.clamp(part.abs().amax(-1) / top, min=1e-12)
        scales[r:r + 64] = s
        codes[r:r + 64] = torch.clamp(torch.round(part / s[..., None]), -127, 127).to(torch.int8).view(torch.uint8)
    return codes, scales


def _layer(case, seed, layer):
    """One layer's inputs of a decode case: history codes and scales, q and the current token."""
    r = _Draw(seed * 64 + layer)
    b, h, d, rows = case["batch"], case["heads"], case["head_dim"], case["batch"] * case["heads"]
    k = _quantized(r.history("k", b, h, case["tokens"], d))
    v = _quantized(r.history("v", b, h, case["tokens"], d))
    return k, v, [r.normal(n, (rows, 1, d), case["q"]) for n in ("q", "sk", "sv")]


def _float_layer(case, seed):
    r = _Draw(seed * 64)
    b, h, d, rows = case["batch"], case["heads"], case["head_dim"], case["batch"] * case["heads"]
    kv = DTYPES[case["kv"]]
    return (r.history("k", b, h, case["tokens"], d).to(kv), r.history("v", b, h, case["tokens"], d).to(kv),
            r.normal("q", (rows, 1, d), case["q"]), r.normal("kn", (rows, d), case["q"]),
            r.normal("vn", (rows, d), case["q"]))


def _append_source(case, seed, layer):
    r = _Draw(seed * 64 + layer)
    shape = (case["batch"], case["heads"], case["tokens"], case["head_dim"])
    return [r.history(n, *shape).reshape(shape).to(DTYPES[case["src"]]) for n in ("k", "v")]


def _append_past(case) -> list[int]:
    rng = random.Random(case["tokens"])
    return [case["past"] + rng.randint(0, case["past"]) for _ in range(case["batch"])]


def _arena_layer(case, seed, layer):
    """One layer's prefill (bf16) and current token of the arena case."""
    r = _Draw(seed * 64 + layer)
    b, h, d = case["batch"], case["heads"], case["head_dim"]
    hist = [r.history(n, b, h, case["tokens"], d).reshape(b, h, case["tokens"], d).bfloat16() for n in ("k", "v")]
    return hist, [r.normal(n, (b * h, 1, d), case["q"]) for n in ("q", "kn", "vn")]


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["op"]](case, seed)


def _prepare_decode(case, seed):
    b, h, d, cap, layers = case["batch"], case["heads"], case["head_dim"], case["capacity"], case["layers"]
    rows = b * h
    lens = lengths_of(case)
    past = torch.tensor(lens, dtype=torch.int32, device=DEVICE)
    kc = torch.zeros((layers, rows, cap, d), dtype=torch.uint8, device=DEVICE)
    vc = torch.zeros_like(kc)
    ks = torch.zeros((layers, rows, cap), dtype=torch.float32, device=DEVICE)
    vs = torch.zeros_like(ks)
    out = torch.empty((layers, rows, 1, d), dtype=DTYPES[case["out"]], device=DEVICE)
    steps = []
    for i in range(layers):
        k, v, (q, sk, sv) = _layer(case, seed, i)
        n = case["tokens"]
        kc[i, :, :n], ks[i, :, :n] = k
        vc[i, :, :n], vs[i, :, :n] = v
        make = ppk.DecodeStep if case["step"] else ppk.DecodeAttention
        steps.append(make(q, kc[i], vc[i], ks[i], vs[i], sk, sv, past, h, bf16_history=case["bf16_history"],
                          max_past=max(lens), out=out[i], past_host=lens if case["host"] else None))
    keep = {"out": out}
    if case["step"]:
        keep.update(k_codes=kc, v_codes=vc, k_scales=ks, v_scales=vs)
    return {"op": "calls", "calls": steps, "outputs": keep}


def _prepare_float(case, seed):
    b, h, d, cap = case["batch"], case["heads"], case["head_dim"], case["capacity"]
    rows, n = b * h, case["tokens"]
    lens = lengths_of(case)
    k, v, q, kn, vn = _float_layer(case, seed)
    ks = torch.zeros((rows, cap, d), dtype=k.dtype, device=DEVICE)
    vs = torch.zeros_like(ks)
    ks[:, :n], vs[:, :n] = k, v
    lengths = torch.tensor(lens, dtype=torch.int32, device=DEVICE)
    out = torch.empty((rows, 1, d), dtype=DTYPES[case["out"]], device=DEVICE)
    host = lens if case["host"] else None
    if case["step"]:
        call = ppk.FloatDecodeStep(q, ks, vs, lengths, h, kn, vn, max_length=max(lens) + 1, out=out,
                                   lengths_host=host)
        return {"op": "calls", "calls": [call], "outputs": {"out": out, "k": ks, "v": vs}}
    call = ppk.FloatDecodeAttention(q, ks, vs, lengths, h, max_length=max(lens), out=out, lengths_host=host)
    return {"op": "calls", "calls": [call], "outputs": {"out": out}}


def _prepare_append(case, seed):
    b, h, d, cap, layers = case["batch"], case["heads"], case["head_dim"], case["capacity"], case["layers"]
    past = torch.tensor(_append_past(case), dtype=torch.int32, device=DEVICE)
    kc = torch.zeros((layers, b * h, cap, d), dtype=torch.uint8, device=DEVICE)
    vc = torch.zeros_like(kc)
    ks = torch.zeros((layers, b * h, cap), dtype=torch.float32, device=DEVICE)
    vs = torch.zeros_like(ks)
    calls = []
    for i in range(layers):
        k, v = _append_source(case, seed, i)
        calls.append(ppk.AppendKV(k, v, past, kc[i], vc[i], ks[i], vs[i]))
    return {"op": "calls", "calls": calls,
            "outputs": {"k_codes": kc, "v_codes": vc, "k_scales": ks, "v_scales": vs}}


def _prepare_codec(case, seed):
    x = _Draw(seed).history("x", 1, case["rows"], case["tokens"], case["head_dim"]).to(DTYPES[case["src"]])
    return {"op": "codec", "x": x, "out": DTYPES[case["out"]]}


def _prepare_arena(case, seed):
    lens = lengths_of(case)
    layers = []
    for i in range(case["layers"]):
        (k, v), (q, kn, vn) = _arena_layer(case, seed, i)
        caches = [LayerCache("int8", case["heads"], case["head_dim"], device=0) for _ in lens]
        for b, (cache, n) in enumerate(zip(caches, lens)):
            cache.query(k[b, :, :n].contiguous(), v[b, :, :n].contiguous(), 0, True)
        # The sequences join into one batch arena; the rounds that follow use it as it is.
        LayerCache.query_batch(caches, None, None, lens, False)
        layers.append((caches, q, kn, vn))
    return {"op": "arena", "layers": layers, "lens": lens, "heads": case["heads"], "head_dim": case["head_dim"]}


def _prepare_sample(case, seed):
    r = _Draw(seed)
    b, g, n = case["batch"], case["guidance"], case["choices"]
    raw = 3.0 * r.normal("raw", (b * g, n))
    uniforms = torch.rand((b, 1), generator=r._gen("uniform"), device=DEVICE)
    count = torch.randint(case["least_legal"], n + 1, (b,), generator=r._gen("count"), device=DEVICE)
    start = (torch.rand((b,), generator=r._gen("start"), device=DEVICE) * (n - count + 1)).long()
    bounds = torch.stack([start, count], 1).to(torch.int32).contiguous()
    call = ppk.RenyiSampler(raw, uniforms, bounds, case["alpha"], case["cfg"], g, 1000)
    return {"op": "calls", "calls": [call], "outputs": {"sample": call.out}}


_PREPARE = {"decode": _prepare_decode, "float": _prepare_float, "append": _prepare_append, "codec": _prepare_codec,
            "arena": _prepare_arena, "sample": _prepare_sample}


def run(state):
    if state["op"] == "calls":
        for call in state["calls"]:
            call()
        return state["outputs"]
    if state["op"] == "codec":
        codes, scales = ppk.quantize(state["x"])
        return {"codes": codes, "scales": scales, "values": ppk.dequantize(codes, scales, state["out"])}
    lens = state["lens"]
    plan = WritePlan(lens, state["heads"], state["head_dim"])
    outs = []
    for caches, q, kn, vn in state["layers"]:
        # An uncommitted round (commit = False): the slot is written and
        # attended, the caches' committed lengths stay.
        view = LayerCache.query_batch(caches, None, None, lens, False, plan)
        outs.append(arena_decode_step(view, q, kn, vn, state["heads"], past_host=lens))
    return {"out": outs}


# ---------------------------------------------------------------------------
# exact: plain torch in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    op = case["op"]
    if op == "sample":
        return None
    if op == "codec":
        x = _Draw(seed).history("x", 1, case["rows"], case["tokens"], case["head_dim"]).to(DTYPES[case["src"]])
        codes, scales = _quantized(x.float())
        s = torch.clamp(x.double().abs().amax(-1) / 127.0, min=1e-12)
        return {"codes": None, "scales": s, "values": codes.view(torch.int8).double() * scales.double()[..., None]}
    if op == "append":
        past, d = _append_past(case), case["head_dim"]
        shape = (case["layers"], case["batch"], case["heads"], case["capacity"])
        got = {"k_codes": None, "v_codes": None}
        for name in ("k_scales", "v_scales"):
            got[name] = torch.zeros(shape, dtype=torch.float64, device=DEVICE)
        for i in range(case["layers"]):
            for name, x in zip(("k_scales", "v_scales"), _append_source(case, seed, i)):
                s = torch.clamp(x.double().abs().amax(-1) / 127.0, min=1e-12)
                for b, p in enumerate(past):
                    got[name][i, b, :, p:p + case["tokens"]] = s[b]
        for name in ("k_scales", "v_scales"):
            got[name] = got[name].reshape(case["layers"], case["batch"] * case["heads"], case["capacity"])
        return got
    lens = lengths_of(case)
    if op == "float":
        k, v, q, kn, vn = _float_layer(case, seed)
        if not case["step"]:
            return {"out": _attend(k, v, q, lens, None, None)}
        cur = [t.to(k.dtype) for t in (kn, vn)]
        return {"out": _attend(k, v, q, lens, *cur), "k": None, "v": None}
    outs = []
    for i in range(case["layers"]):
        if op == "arena":
            hist, (q, sk, sv) = _arena_layer(case, seed, i)
            (kc, ks), (vc, vs) = [_quantized(x.float().reshape(-1, case["tokens"], case["head_dim"])) for x in hist]
        else:
            (kc, ks), (vc, vs), (q, sk, sv) = _layer(case, seed, i)
        hist = (kc, ks, vc, vs)
        outs.append(_attend_int8(hist, q, sk, sv, lens, case.get("bf16_history", False)))
    if op == "arena":
        return {"out": outs}
    got = {"out": torch.stack(outs)}
    if case["step"]:
        got.update(k_codes=None, v_codes=None, k_scales=None, v_scales=None)
    return got


def _attend_int8(hist, q, sk, sv, lens, bf16_history):
    kc, ks, vc, vs = hist

    def widen(codes, scales):
        if bf16_history:  # each element is the bf16 rounding of the f32 product
            return (codes.view(torch.int8).float() * scales[..., None]).bfloat16().double()
        return codes.view(torch.int8).double() * scales.double()[..., None]

    out, heads = [], q.shape[0] // len(lens)
    for b in range(len(lens)):
        r = slice(b * heads, (b + 1) * heads)
        out.append(_attend(widen(kc[r], ks[r]), widen(vc[r], vs[r]), q[r], [lens[b]], sk[r], sv[r]))
    return torch.cat(out)


def _attend(k, v, q, lens, sk, sv):
    """softmax(q . [k, sk] / sqrt(d)) . [v, sv] in 64 bits, sequence by sequence."""
    rows, _, d = q.shape
    heads = rows // len(lens)
    out = torch.empty((rows, 1, d), dtype=torch.float64, device=q.device)
    for b, n in enumerate(lens):
        r = slice(b * heads, (b + 1) * heads)
        kk, vv, qq = k[r, :n].double(), v[r, :n].double(), q[r].double()
        if sk is not None:
            kk = torch.cat([kk, sk[r].double().reshape(heads, 1, d)], 1)
            vv = torch.cat([vv, sv[r].double().reshape(heads, 1, d)], 1)
        p = torch.softmax((kk * qq).sum(-1) / math.sqrt(d), -1)
        out[r] = (p[..., None] * vv).sum(1, keepdim=True)
    return out


def tolerance(case):
    op = case["op"]
    if op in ("append", "codec", "sample"):
        return "exact"  # codes, scales, dequantised values and tokens are defined bit for bit
    if case.get("out", "f32") == "bf16":
        return {"rel": 2e-3, "max": 0.01}  # one rounding to 8 bits
    return {"rel": 1e-5, "max": 5e-4}  # f32 sums in another order (a few 1e-7 as measured; heavy channels nearly cancel)
