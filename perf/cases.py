"""The calls whose time this library answers for, as plain data, and how each is prepared, run and checked.

Five kinds of call, each through the package's own entry points:

* ``decode``: the attention of one decode token over one cache layer
  (``mu_zero_decode_attention_forward``), the call a model makes per layer and step.
* ``prefill``: a prompt's K / V taken in by a new cache layer (``MuZeroCacheLayer.update``): alpha
  selection, quantization, packing.
* ``dense``: the whole cache of a layer as dense K / V (``MuZeroCacheLayer.dense_kv``), what chunked
  prefill, cropping and attention implementations without the decode hook read.
* ``codec``: ``roundtrip``, the offline quantize + dequantize of one K and one V tensor.
* ``stream``: one layer's part of a generation: prefill, then decode steps, each the fused prologue (q/k
  norm, rotary embedding, residual append), the flush when it is due, and the decode attention.

Inputs are N(0, 1) with four key channels ten times larger, as keys with outlier channels are.
"""

import math

import torch

from muzero_amd import MuZeroCacheLayer, MuZeroConfig, mu_zero_decode_attention_forward, roundtrip
from muzero_amd.kernels import loader

GROUP = 64
EPS = 1e-8
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
META = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
# (query heads, kv heads, head_dim) of the attention layers that the tests and the benchmark name
SHAPES = ((32, 8, 128), (28, 4, 128), (40, 8, 128), (64, 8, 128), (16, 8, 128), (32, 8, 64), (32, 8, 96))


def _case(name, kind, bits, batch, tokens, shape=(32, 8, 128), io="bf16", meta="float16", residual=128, steps=0,
          alpha_key=2.0, alpha_value=2.0, padded=False):
    case = {"name": name} if name else {}
    case.update(kind=kind, bits=bits, batch=batch, tokens=tokens, q_heads=shape[0], kv_heads=shape[1], head_dim=shape[2],
                io=io, meta=meta, residual=residual, steps=steps, alpha_key=alpha_key, alpha_value=alpha_value,
                padded=padded)
    return case


def listed():
    return [
        # one user's chat turn: the smallest call, all latency
        _case("decode_b1_c1k_4bit", "decode", 4, 1, 1000),
        # the benchmark's batch-serving step
        _case("decode_b64_c4k_4bit", "decode", 4, 64, 4096),
        # the quality-first width, with the two alphas that keys with outlier channels get
        _case("decode_b64_c4k_8bit", "decode", 8, 64, 4096, alpha_key=4.0),
        # long documents: few sequences, many tokens, the split over tokens
        _case("decode_b8_c32k_2bit", "decode", 2, 8, 32768),
        # a small model's heads (head_dim 64) at a ragged length
        _case("decode_b24_c3001_hd64_4bit", "decode", 4, 24, 3001, shape=(32, 8, 64)),
        # a left-padded batch of prompts of different lengths, seven query heads per kv-head, fp16
        _case("decode_b12_c2777_3bit_padded", "decode", 3, 12, 2777, shape=(28, 4, 128), io="f16", padded=True),
        # head_dim 96: the separate qk and av launches behind the same hook
        _case("decode_b8_c2k_hd96_4bit", "decode", 4, 8, 2100, shape=(32, 8, 96)),
        # the benchmark's prompts entering the cache
        _case("prefill_b64_c4k_4bit", "prefill", 4, 64, 4096),
        # an fp16 model's shorter prompts, alphas chosen from the data
        _case("prefill_b16_c2k_8bit_f16", "prefill", 8, 16, 2000, io="f16", alpha_key=0.0, alpha_value=0.0),
        # a chunked prefill's read of what is already cached
        _case("dense_b16_c4k_4bit", "dense", 4, 16, 4096),
        # the offline quality check of one small K and V
        _case("codec_b1_c896_4bit", "codec", 4, 1, 896),
        # a batch generating through one flush, alphas chosen from the data (2 at this width)
        _case("stream_b32_c4k_2bit", "stream", 2, 32, 4136, steps=40, alpha_key=0.0, alpha_value=0.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode",) * 6 + ("prefill",) * 3 + ("dense", "codec", "stream"))
    bits = rng.choice((1, 2, 3, 4, 4, 4, 7, 8))
    alpha_key = 4.0 if bits == 8 else rng.choice((4.0, 16.0)) if bits == 1 else 2.0  # as the rules give such keys
    alpha_value = 4.0 if bits == 3 and rng.random() < 0.5 else 2.0
    io = rng.choice(("bf16", "bf16", "bf16", "f16"))
    meta = rng.choice(("float16", "float16", "float16", "bfloat16", "float32"))
    shape = rng.choice(SHAPES[:1] * 4 + SHAPES[1:])
    residual = rng.choice((64, 128, 128, 128, 256))
    batch = _log(rng, 1, 128)
    if kind == "decode":
        # at most the tokens of 64 sequences of 4096, kv-heads and head_dim as the benchmark's
        most = 64 * 4096 * 8 * 128 // (batch * shape[1] * shape[2])
        tokens = min(most, _log(rng, 200, 32768))
        return _case("", kind, bits, batch, max(tokens, 200), shape, io, meta, residual, 0, alpha_key, alpha_value,
                     padded=rng.random() < 0.25)
    if kind == "prefill":
        io = rng.choice(("bf16", "bf16", "f16", "f32"))
        tokens = min(_log(rng, 200, 16384), (96 if io == "f32" else 192) * 1024 // batch)
        given = rng.random() < 0.3  # alphas preset by the configuration instead of chosen from the data
        return _case("", kind, bits, batch, max(tokens, 200), shape, io, meta, residual, 0,
                     alpha_key if given else 0.0, alpha_value if given else 0.0)
    if kind == "dense":
        tokens = min(_log(rng, 200, 16384), 64 * 1024 // batch)
        return _case("", kind, bits, batch, max(tokens, 200), shape, io, meta, residual, 0, alpha_key, alpha_value)
    if kind == "codec":
        batch = _log(rng, 1, 8)
        io = rng.choice(("bf16", "f16", "f32"))
        return _case("", kind, bits, batch, GROUP * _log(rng, 1, 64), shape[:2] + (rng.choice((64, 96, 128)),), io, meta,
                     0, 0, alpha_key, alpha_value)
    shape = rng.choice(SHAPES[:6])  # the prologue serves head_dim 64 and 128
    batch = _log(rng, 1, 48)
    tokens = min(_log(rng, 200, 8192), 128 * 1024 // batch)
    return _case("", kind, bits, batch, max(tokens, 200), shape, io, meta, 128, rng.randint(8, 48), alpha_key, alpha_value)


# --------------------------------------------------------------------------- inputs

def _generator(case, seed):
    return torch.Generator(device="cuda").manual_seed(7919 * seed + case["batch"] + 131 * case["tokens"])


def _randn(shape, dtype, g):
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for row in out:  # one batch row at a time: no fp32 copy of the whole tensor
        row.copy_(torch.randn(row.shape, generator=g, device="cuda"))
    return out


def _kv(case, tokens, g):
    dtype, shape = DTYPES[case["io"]], (case["batch"], case["kv_heads"], tokens, case["head_dim"])
    k, v = _randn(shape, dtype, g), _randn(shape, dtype, g)
    k[..., torch.randperm(case["head_dim"], generator=g, device="cuda")[:4]] *= 10.0
    return k, v


def _mask(case, length, g):
    """Left padding of up to a third of the prompt, as the additive mask that transformers builds."""
    if not case["padded"]:
        return None
    dtype = DTYPES[case["io"]]
    pad = torch.randint(0, length // 3 + 1, (case["batch"],), generator=g, device="cuda")
    pad[0] = 0
    hidden = torch.arange(length, device="cuda")[None] < pad[:, None]
    mask = torch.zeros(case["batch"], length, dtype=dtype, device="cuda")
    return mask.masked_fill_(hidden, torch.finfo(dtype).min)[:, None, None, :]


def _config(case):
    return MuZeroConfig(bits=case["bits"], residual_length=case["residual"], amax_dtype=case["meta"],
                        alpha_key=case["alpha_key"] or None, alpha_value=case["alpha_value"] or None)


class _Attention:
    """What the decode hook reads from a model's attention module."""

    training = False

    def __init__(self, case):
        self.num_key_value_groups = case["q_heads"] // case["kv_heads"]


def _stream_inputs(case, g):
    """Per-step projections, rotary rows and norm weights of one layer."""
    dtype, d, n = DTYPES[case["io"]], case["head_dim"], case["steps"]
    heads = (case["q_heads"], case["kv_heads"], case["kv_heads"])
    q, k, v = (_randn((n, case["batch"], h, d), dtype, g) for h in heads)
    k[..., torch.randperm(d, generator=g, device="cuda")[:4]] *= 10.0
    inv = 1e6 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float32) / d)
    angle = (case["tokens"] + torch.arange(n, device="cuda", dtype=torch.float32))[:, None] * inv
    angle = torch.cat([angle, angle], dim=-1)
    weights = [(1.0 + 0.1 * torch.randn(d, generator=g, device="cuda")).to(dtype) for _ in range(2)]
    return q, k, v, angle.cos().to(dtype)[:, None], angle.sin().to(dtype)[:, None], weights


def _raw(case, seed):
    """Every input of the case, from the seed alone."""
    g = _generator(case, seed)
    k, v = _kv(case, case["tokens"], g)
    if case["kind"] == "decode":
        q = _randn((case["batch"], case["q_heads"], 1, case["head_dim"]), DTYPES[case["io"]], g)
        return k, v, q, _mask(case, case["tokens"], g)
    if case["kind"] == "stream":
        return (k, v) + _stream_inputs(case, g)
    return k, v


def _filled(case, k, v):
    """A layer that has taken in the prompt, its last token as a decode step."""
    layer = MuZeroCacheLayer(_config(case))
    layer.update(k[:, :, :-1], v[:, :, :-1])
    layer.update(k[:, :, -1:], v[:, :, -1:], {"materialize_full_kv": False})
    return layer


def prepare(case, seed):
    raw = _raw(case, seed)
    state = {"case": case, "scaling": case["head_dim"] ** -0.5, "module": _Attention(case)}
    if case["kind"] == "decode":
        state.update(layer=_filled(case, raw[0], raw[1]), query=raw[2], mask=raw[3])
    elif case["kind"] == "dense":
        state.update(layer=_filled(case, *raw))
    elif case["kind"] == "stream":
        state.update(zip(("k", "v", "q_new", "k_new", "v_new", "cos", "sin", "norms"), raw))
    else:
        state.update(k=raw[0], v=raw[1])
    return state


# --------------------------------------------------------------------------- one pass

def _stored(layer):
    out = {"key_codes": layer._packed_key_q, "key_min": layer._key_mn, "key_scale": layer._key_scale,
           "value_codes": layer._packed_value_q, "value_min": layer._value_mn, "value_scale": layer._value_scale,
           "keys": layer.keys, "values": layer.values}
    return {name: t for name, t in out.items() if t is not None}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        layer = state["layer"]
        return mu_zero_decode_attention_forward(state["module"], state["query"], state["mask"], state["scaling"],
                                                layer.get_attention_state())[0]
    if kind == "prefill":
        layer = MuZeroCacheLayer(_config(case))
        layer.update(state["k"], state["v"])
        return dict(_stored(layer), alphas=[layer._selected_alpha_key or 0.0, layer._selected_alpha_value or 0.0])
    if kind == "dense":
        return state["layer"].dense_kv()
    if kind == "codec":
        return roundtrip(state["k"], state["v"], bits=case["bits"], alpha_key=case["alpha_key"],
                         alpha_value=case["alpha_value"], amax_dtype=META[case["meta"]])
    layer = MuZeroCacheLayer(_config(case))
    layer.update(state["k"], state["v"])
    outs = []
    for t in range(case["steps"]):
        k_row, v_row = layer.decode_append_slot()
        query = loader.decode_prologue(state["q_new"][t], state["k_new"][t], state["v_new"][t], state["cos"][t],
                                       state["sin"][t], *state["norms"], 1e-6, k_row[:, :, 0], v_row[:, :, 0])
        layer.decode_append_commit()
        outs.append(mu_zero_decode_attention_forward(state["module"], query, None, state["scaling"],
                                                     layer.get_attention_state())[0])
    return {"steps": outs, "stored": _stored(layer)}


# --------------------------------------------------------------------------- what a pass cannot do without

def _prefix(case, tokens):
    """Quantized tokens of `tokens`: whole groups above the residual window."""
    return max(tokens - case["residual"], 0) // GROUP * GROUP


def _packed_bytes(case, tokens):
    """Codes and min / scale of `tokens` quantized K and V tokens of every head."""
    meta = 8 if case["meta"] == "float32" else 4
    per_group = 8 * case["bits"] + meta
    heads, d = case["batch"] * case["kv_heads"], case["head_dim"]
    return heads * (tokens // GROUP) * d * per_group + heads * tokens * -(-d // GROUP) * per_group


def _dense_bytes(case, tokens):
    return 2 * case["batch"] * case["kv_heads"] * tokens * case["head_dim"] * DTYPES[case["io"]].itemsize


def _decode_work(case, tokens):
    lq = _prefix(case, tokens)
    qo = 2 * case["batch"] * case["q_heads"] * case["head_dim"] * DTYPES[case["io"]].itemsize
    mask = case["batch"] * tokens * DTYPES[case["io"]].itemsize if case["padded"] else 0
    return (_packed_bytes(case, lq) + _dense_bytes(case, tokens - lq) + qo + mask,
            4 * case["batch"] * case["q_heads"] * tokens * case["head_dim"])


def work(case):
    tokens = case["tokens"]
    values = 2 * case["batch"] * case["kv_heads"] * tokens * case["head_dim"]
    lq = _prefix(case, tokens)
    if case["kind"] == "decode":
        nbytes, flops = _decode_work(case, tokens)
    elif case["kind"] == "prefill":  # the prompt read, the prefix written; about ten operations a value
        nbytes, flops = _dense_bytes(case, tokens) + _packed_bytes(case, lq), 10 * values
    elif case["kind"] == "dense":  # the prefix and the residual read, dense K / V written; four operations a value
        nbytes, flops = _packed_bytes(case, lq) + _dense_bytes(case, tokens - lq) + _dense_bytes(case, tokens), 4 * values
    elif case["kind"] == "codec":  # in and out: the codes need not leave the chip
        nbytes, flops = 2 * _dense_bytes(case, tokens), 14 * values
    else:
        nbytes, flops = _dense_bytes(case, tokens) + _packed_bytes(case, lq), 10 * values
        for t in range(1, case["steps"] + 1):
            b, f = _decode_work(case, tokens + t)
            row = _dense_bytes(case, 1)
            nbytes, flops = nbytes + b + 2 * row, flops + f
    return {"bytes": nbytes, "flops": flops}


# --------------------------------------------------------------------------- how far results may differ

def tolerance(case):
    """Codes, min / scale and dequantized values are fixed bit for bit (the reference quantizer's
    operations in the input's type), attention is not: its sums may be taken in any order."""
    if case["kind"] in ("prefill", "dense", "codec"):
        return "exact"
    # about four times the error against 64 bits that was measured (bf16 0.0017, fp16 0.0002: the outputs' own rounding)
    rel = {"bf16": 0.007, "f16": 0.001}[case["io"]]
    if case["head_dim"] not in (64, 128):
        rel *= 4  # the separate launches round logits and weights to the query's type between the steps (bf16 0.012)
    elif case["head_dim"] == 64 or case["bits"] == 7:
        rel *= 3  # values may be held in fp32 or rounded to the layer's type (bf16 0.006)
    return {"rel": rel}


# --------------------------------------------------------------------------- the same in 64 bits

def _quantize(rows, bits, alpha, meta):
    """Codes, min and scale of rows [N, 64]: the quantizer's definition, each operation in the rows' type."""
    top = float((1 << bits) - 1)
    lo, hi = rows.amin(-1, keepdim=True), rows.amax(-1, keepdim=True)
    span = (hi - lo).clamp_min(EPS)
    unit, zero = ((rows - lo) / span).clamp(0.0, 1.0), ((0.0 - lo) / span).clamp(0.0, 1.0)
    level = torch.round(zero * top)
    base = torch.log1p(torch.tensor(alpha, dtype=torch.float32, device=rows.device))

    def steps(distance, extent, bins):
        p = (distance / extent.clamp_min(EPS)).clamp(0.0, 1.0)
        share = (torch.log1p(alpha * p).float() / base).to(rows.dtype)  # base is not rounded to the rows' type
        return torch.round(share * bins.clamp_min(1.0))

    up, down = steps(unit - zero, 1.0 - zero, top - level), steps(zero - unit, zero, level)
    codes = torch.where(unit >= zero, level + up, level - down).clamp(0.0, top)
    return codes, lo.to(meta), span.to(meta)


def _dequantize(codes, lo, span, bits, alpha):
    """float64 values of the codes, from min and scale as stored (the zero level in fp32, as it is defined)."""
    top = float((1 << bits) - 1)
    q, lo32, span32 = codes.double(), lo.float(), span.float().clamp_min(EPS)
    zero32 = ((0.0 - lo32) / span32).clamp(0.0, 1.0)
    level = torch.round(zero32 * top).double()
    lo, span, zero = lo32.double(), span32.double(), zero32.double()
    base = math.log1p(alpha)
    up = torch.expm1(((q - level) / (top - level).clamp_min(1.0)).clamp(0.0, 1.0) * base) / alpha
    down = torch.expm1(((level - q) / level.clamp_min(1.0)).clamp(0.0, 1.0) * base) / alpha
    unit = torch.where(q >= level, zero + (1.0 - zero) * up, zero - zero * down).clamp(0.0, 1.0)
    return unit * span + lo


def _through(block, kind, case, alpha, rows_type=None):
    """[H, T, D] of one batch row through the quantizer and back, float64."""
    h, t, d = block.shape
    if kind == "key":
        rows = block.reshape(h, t // GROUP, GROUP, d).transpose(2, 3).reshape(-1, GROUP)
    else:
        rows = torch.nn.functional.pad(block, (0, -d % GROUP)).reshape(-1, GROUP)
    rows = rows if rows_type is None else rows.to(rows_type)
    x = _dequantize(*_quantize(rows, case["bits"], alpha, META[case["meta"]]), case["bits"], alpha)
    if kind == "key":
        return x.reshape(h, t // GROUP, d, GROUP).transpose(2, 3).reshape(h, t, d)
    return x.reshape(h, t, -1)[..., :d]


def _dense_row(k, v, lq, case):
    """One batch row's K and V, float64: the prefix through the quantizer, in the layer's type as the cache holds it."""
    alphas = case["alpha_key"] or 2.0, case["alpha_value"] or 2.0
    both = []
    for x, kind, alpha in ((k, "key", alphas[0]), (v, "value", alphas[1])):
        head = _through(x[:, :lq], kind, case, alpha).to(x.dtype).double() if lq else x[:, :0].double()
        both.append(torch.cat([head, x[:, lq:].double()], 1))
    return both


def _attend(q, k, v, mask, scaling):
    """[Hq, D] of one batch row."""
    hq, d = q.shape
    logits = torch.matmul(q.double().reshape(k.shape[0], -1, d), k.transpose(1, 2).contiguous()) * scaling
    if mask is not None:
        logits = logits + mask.double()
    return torch.matmul(torch.softmax(logits, -1), v).reshape(hq, d)


def _rotate(x, weight, cos, sin):
    """The norm and rotary embedding of a projection [H, D], rounded where a model in this type rounds."""
    f = x.float()
    x = weight * (f * torch.rsqrt(f.square().mean(-1, keepdim=True) + 1e-6)).to(x.dtype)
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def exact(case, seed):
    if case["kind"] == "prefill":
        return None  # bytes, and minima and ranges rounded to the metadata's type
    raw = _raw(case, seed)
    k, v = raw[:2]
    scaling, kind = case["head_dim"] ** -0.5, case["kind"]
    if kind == "codec":
        return [torch.stack([_through(row, name, case, case["alpha_" + name], torch.float32) for row in x])
                for x, name in ((k, "key"), (v, "value"))]
    lq = _prefix(case, case["tokens"])
    if kind == "dense":
        rows = [[_through(x[b, :, :lq], name, case, case["alpha_" + name]) if lq else x[b, :, :0].double()
                 for b in range(case["batch"])] for x, name in ((k, "key"), (v, "value"))]
        return [torch.cat([torch.stack(r), x[:, :, lq:].double()], 2) for r, x in zip(rows, (k, v))]
    if kind == "decode":
        q, mask = raw[2:]
        out = []
        for b in range(case["batch"]):
            dk, dv = _dense_row(k[b], v[b], lq, case)
            out.append(_attend(q[b, :, 0], dk, dv, None if mask is None else mask[b, 0], scaling))
        return torch.stack(out)[:, None]
    if case["batch"] * case["tokens"] * case["steps"] > 6_000_000:
        return None  # more than seconds in 64 bits
    q_new, k_new, v_new, cos, sin, norms = raw[2:]
    steps = [[] for _ in range(case["steps"])]
    for b in range(case["batch"]):
        kb, vb, last, dense = k[b], v[b], -1, None
        for t in range(case["steps"]):
            kb = torch.cat([kb, _rotate(k_new[t, b], norms[1], cos[t, 0], sin[t, 0])[:, None]], 1)
            vb = torch.cat([vb, v_new[t, b][:, None]], 1)
            lq = _prefix(case, kb.shape[1])
            dense = _dense_row(kb, vb, lq, case) if lq != last else [torch.cat([x, y[:, -1:].double()], 1)
                                                                     for x, y in zip(dense, (kb, vb))]
            last = lq
            steps[t].append(_attend(_rotate(q_new[t, b], norms[0], cos[t, 0], sin[t, 0]), *dense, None, scaling))
    return {"steps": [torch.stack(rows)[:, None] for rows in steps], "stored": None}
