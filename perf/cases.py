"""The work this framework is timed on: what an encoder or decoder of TSAC
streams has it do, from one projection of one frame step to a whole recording.

Sizes are those of the benchmark and the tests: 30 s of 44.1 kHz audio is 2584
frames of 512 samples (2580 as a token stream), 12 codebooks of stereo or 9 of
mono, coded in up to a few lanes (the entropy batch); the probability model is
the reference geometry (width 512, 4 x 128 heads, FFN 2048) or the wide one
(width 1024, 16 x 64 heads, FFN 4096), 12 temporal and 3 codebook layers.
Weights are seeded and random, tokens uniform over the alphabet, audio is sines
plus noise.

Every result is compared bit for bit. A stream can only be decoded where the
decoder's probabilities equal the encoder's in every bit, so every operator has
one fixed order of operations and its tests compare bits; tokens, streams and
PCM follow from those.
"""
import math
import os
import sys

import numpy as np
import torch

PACKAGE = os.path.join(os.getcwd(), "tsac-metal_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

from tsac_hip import native, synthetic  # noqa: E402

GEOMETRIES = {"reference": synthetic.REFERENCE, "wide": synthetic.WIDE}
#: A small model for the codec's own calls, which need a session but run no model.
SESSION_GEOMETRY = synthetic.Geometry(width=256, heads=2, head_width=128, ffn=512, temporal_layers=1,
                                      codebook_layers=1, latent=256)
HOP = 512


def listed():
    return [
        # One projection of one decoded frame in three lanes, through the operator
        # entry point: the smallest call, mostly launches and waiting.
        {"name": "linear_step", "kind": "linear", "rows": 3, "K": 1024, "N": 4096},
        # One new frame's attention over a nearly full context, three lanes.
        {"name": "attention_step", "kind": "attention_step", "sequences": 3, "time": 1021, "heads": 16,
         "head_width": 64},
        # The feed-forward block over one second of stereo (87 frames x 12 codebooks).
        {"name": "mlp_clip", "kind": "mlp", "rows": 1044, "geometry": "reference"},
        # The same block over every token of 30 s at the wide geometry.
        {"name": "mlp_encode", "kind": "mlp", "rows": 30960, "geometry": "wide"},
        # The model's head over 10 s (862 frames x 12 codebooks): final norm, logits, probabilities.
        {"name": "head_encode", "kind": "head", "rows": 10344, "geometry": "reference"},
        # Causal self-attention of the known frames of 30 s in three lanes.
        {"name": "attention_encode", "kind": "attention_causal", "lengths": "862,861,861", "heads": 16,
         "head_width": 64},
        # Codec synthesis of one second of mono: few frames for deep layers.
        {"name": "synthesis_clip", "kind": "synthesis", "frames": 87, "channels": 1, "books": 9},
        # Codec synthesis of 30 s of stereo.
        {"name": "synthesis_track", "kind": "synthesis", "frames": 2584, "channels": 2, "books": 12},
        # A 30 s stereo recording from PCM to its stream: codec analysis, the model
        # over all tokens, range coding.
        {"name": "audio_encode", "kind": "audio_encode", "samples": 1323000, "channels": 2, "books": 12, "batch": 3},
        # The wide model and range coder over the tokens of 30 s.
        {"name": "model_encode", "kind": "model_encode", "frames": 2580, "books": 12, "batch": 3, "geometry": "wide"},
        # The wide model decoding 9 s in three lanes, frame step by frame step.
        {"name": "model_decode", "kind": "model_decode", "frames": 774, "books": 12, "batch": 3, "geometry": "wide"},
        # A 30 s stereo stream back to PCM: frame steps, then codec synthesis.
        {"name": "audio_decode", "kind": "audio_decode", "frames": 2584, "channels": 2, "books": 12, "batch": 3},
    ]


def _spread(rng, low, high):
    """A whole number, uniform in its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "attention_step", "attention_step", "mlp", "mlp", "head",
                       "attention_causal", "attention_causal", "synthesis", "synthesis", "analysis",
                       "model_encode", "model_decode", "audio_encode", "audio_decode"])
    geometry = rng.choice(["reference", "wide"])
    g = GEOMETRIES[geometry]
    if kind == "linear":
        return {"kind": kind, "rows": _spread(rng, 1, 30960), "K": rng.choice([512, 1024, 2048, 4096]),
                "N": rng.choice([512, 1024, 1536, 2048, 3072, 4096])}
    if kind == "attention_step":
        return {"kind": kind, "sequences": rng.randint(1, 8), "time": _spread(rng, 1, 2580), "heads": g.heads,
                "head_width": g.head_width}
    if kind in ("mlp", "head"):
        return {"kind": kind, "rows": _spread(rng, 1, 30960), "geometry": geometry}
    if kind == "attention_causal":
        longest = _spread(rng, 1, 1024)
        lengths = [max(1, longest - rng.randint(0, 1 + longest // 8)) for _ in range(rng.randint(1, 3))]
        return {"kind": kind, "lengths": ",".join(str(n) for n in [longest] + lengths), "heads": g.heads,
                "head_width": g.head_width}
    channels = rng.choice([1, 2])
    books = rng.randint(1, 9 if channels == 1 else 12)
    if kind in ("synthesis", "analysis"):
        return {"kind": kind, "frames": _spread(rng, 1, 2584), "channels": channels, "books": books}
    if kind == "model_encode":
        frames = _spread(rng, 3, 2580)
        return {"kind": kind, "frames": frames, "books": books, "batch": rng.randint(1, 3), "geometry": geometry}
    if kind == "model_decode":
        batch = rng.randint(1, 3)
        return {"kind": kind, "frames": _spread(rng, 3, 258 * batch), "books": books, "batch": batch,
                "geometry": geometry}
    if kind == "audio_encode":
        return {"kind": kind, "samples": _spread(rng, 300, 1323000), "channels": channels, "books": books,
                "batch": rng.randint(1, 3)}
    batch = rng.randint(1, 3)
    return {"kind": kind, "frames": _spread(rng, 3, 400 * batch), "channels": channels, "books": books,
            "batch": batch}


# ---------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(1000 + seed)


def _bits(values):
    """BF16 bits of a float tensor, as the operators take them."""
    return values.to(torch.bfloat16).contiguous().view(torch.int16)


def _normal(seed, salt, shape, scale=1.0):
    return _bits(torch.randn(shape, generator=_generator(31 * seed + salt), device="cuda") * scale)


def _blank(*shape):
    return torch.empty(shape, dtype=torch.int16, device="cuda")


def _numbers(bits):
    return bits.view(torch.bfloat16)


def _lengths(case):
    return [int(n) for n in case["lengths"].split(",")]


def _weights(case, seed):
    """The projections an operator case multiplies by: (values, scales, bias) each."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "linear":
        shapes = [(case["K"], case["N"])]
    else:
        g = GEOMETRIES[case["geometry"]]
        shapes = [(g.width, g.ffn), (g.ffn, g.width)] if case["kind"] == "mlp" else [(g.width, g.alphabet)]
    return [synthetic.random_linear(rng, k, n) for k, n in shapes]


def _norm(case, seed):
    width = GEOMETRIES[case["geometry"]].width
    gain = _bits(1.0 + 0.1 * torch.randn(width, generator=_generator(31 * seed + 5), device="cuda"))
    return gain, _normal(seed, 6, (width,), 0.1)


def _rotations(head_width, context):
    table = synthetic.rotary_table(synthetic.Geometry(head_width=head_width, context=context))
    return torch.from_numpy(table.view(np.int16)).cuda()


def _audio(samples, channels, seed):
    """Three sines per channel and low-passed noise, in steps of 16-bit PCM."""
    rng = np.random.default_rng(seed)
    t = np.arange(samples) / 44100.0
    out = np.zeros((samples, channels))
    for c in range(channels):
        for _ in range(3):
            out[:, c] += 0.25 * np.sin(2 * np.pi * rng.uniform(80, 4000) * t + rng.uniform(0, 2 * np.pi))
        noise = rng.standard_normal(samples + 15)
        out[:, c] += 0.2 * np.convolve(noise, np.ones(16) / 4, mode="valid")
    out *= 0.99 / max(1.0, np.abs(out).max())
    return (np.round(out * 32767) / 32768).astype(np.float32)


def _tokens(case, seed):
    return synthetic.random_tokens(case["frames"], 1, case["books"], seed)


def _geometry(case):
    g = GEOMETRIES[case.get("geometry", "reference")]
    if case.get("channels", 2) == 1:
        return synthetic.Geometry(width=g.width, heads=g.heads, head_width=g.head_width, ffn=g.ffn, books=9,
                                  channels=1)
    return g


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear", "mlp", "head"):
        linears = [native.DeviceLinear(*w) for w in _weights(case, seed)]
        rows = case["rows"]
        state = {"kind": kind, "rows": rows, "linears": linears, "x": _normal(seed, 1, (rows, linears[0].K)),
                 "y": _blank(rows, linears[-1].N)}
        if kind != "linear":
            state["gain"], state["bias"] = _norm(case, seed)
            state["normal"] = _blank(rows, linears[0].K)
            state["hidden"] = _blank(rows, linears[0].N)
        if kind == "mlp":
            state["active"] = _blank(rows, linears[0].N)
            state["down"] = _blank(rows, linears[1].N)
        return state
    if kind == "attention_step":
        n, t, w = case["sequences"], case["time"], case["heads"] * case["head_width"]
        return dict(case, query=_normal(seed, 1, (n, w)), keys=_normal(seed, 2, (n, t, w)),
                    values=_normal(seed, 3, (n, t, w)), out=_blank(n, w))
    if kind == "attention_causal":
        lengths, w = _lengths(case), case["heads"] * case["head_width"]
        start = np.cumsum([0] + lengths[:-1])
        ints = [torch.tensor(list(a), dtype=torch.int32, device="cuda") for a in (start, lengths, [0] * len(lengths))]
        return dict(case, qkv=_normal(seed, 1, (sum(lengths), 3 * w)), start=ints[0], length=ints[1], replay=ints[2],
                    sequences=len(lengths), longest=max(lengths), out=_blank(sum(lengths), w),
                    rotations=_rotations(case["head_width"], 1024))
    state = dict(case)
    if kind in ("synthesis", "analysis"):
        model = synthetic.random_model(SESSION_GEOMETRY, 1)
    else:
        model = synthetic.random_model(_geometry(case), seed)
    state["session"] = native.HipModel(model).session()
    if "channels" in case:
        state["dac"] = native.HipDac(synthetic.random_dac(case["channels"], 12 if case["channels"] == 2 else 9, seed))
    if kind == "synthesis":
        state["tokens"] = _tokens(case, seed)
    elif kind == "analysis":
        state["pcm"] = _audio(case["frames"] * HOP, case["channels"], seed)
    elif kind == "audio_encode":
        state["pcm"] = _audio(case["samples"], case["channels"], seed)
    elif kind == "audio_decode":
        header = native.audio_header(case["frames"] * HOP, case["channels"], codebooks=case["books"],
                                     entropy_batch=case["batch"])
        state["stream"] = state["session"].encode(header, _tokens(case, seed))
    else:
        state["header"] = native.header(case["frames"], case["batch"], 1, case["books"])
        state["tokens"] = _tokens(case, seed)
        if kind == "model_decode":
            state["stream"] = state["session"].encode(state["header"], state["tokens"])
    return state


# ---------------------------------------------------------------- one pass

def _stream(data, tokens):
    """A stream, as long as its data makes it, in a buffer for the longest one (ten decisions of up to 16 bits a token)."""
    out = np.zeros(64 + 20 * tokens, np.uint8)
    out[:len(data)] = np.frombuffer(data, np.uint8)
    return {"length": len(data), "stream": out}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        state["linears"][0].apply(state["x"], state["y"])
        return _numbers(state["y"])
    if kind in ("mlp", "head"):
        rows, first = state["rows"], state["linears"][0]
        native.layer_norm(state["x"], rows, first.K, state["gain"], state["bias"], state["normal"])
        first.apply(state["normal"], state["hidden"])
        if kind == "head":
            native.softmax(state["hidden"], rows, first.N, state["y"])
            return _numbers(state["hidden"]), _numbers(state["y"])
        native.gelu(state["hidden"], state["active"])
        state["linears"][1].apply(state["active"], state["down"])
        native.add(state["x"], state["down"], rows, first.K, rows, state["y"])
        return _numbers(state["y"])
    if kind == "attention_step":
        w = state["heads"] * state["head_width"]
        native.attention(state["query"], state["keys"], state["values"], state["time"] * w, state["sequences"],
                         state["time"], state["heads"], state["head_width"], 1 / math.sqrt(state["head_width"]), False,
                         state["out"])
        return _numbers(state["out"])
    if kind == "attention_causal":
        native.attention_causal(state["qkv"], state["heads"], state["head_width"], state["start"], state["length"],
                                state["replay"], state["sequences"], state["longest"], state["rotations"],
                                1 / math.sqrt(state["head_width"]), state["out"])
        return _numbers(state["out"])
    session = state["session"]
    if kind == "synthesis":
        return state["dac"].synthesize(session, state["tokens"], state["frames"], 1, state["books"])
    if kind == "analysis":
        return state["dac"].analyze(session, state["pcm"], state["frames"], 1, state["books"])
    if kind == "audio_encode":
        stream = state["dac"].encode(session, state["pcm"], state["channels"], codebooks=state["books"],
                                     entropy_batch=state["batch"])
        return _stream(stream, -(-len(state["pcm"]) // HOP) * state["books"])
    if kind == "audio_decode":
        return state["dac"].decode(session, state["stream"])[0]
    if kind == "model_encode":
        return _stream(session.encode(state["header"], state["tokens"]), len(state["tokens"]))
    return session.decode(state["stream"])


# ---------------------------------------------------------------- work

def _linear_bytes(k, n):
    return k * n + 4 * (k // 256) * n + 4 * n


def _convolutions(synthesis, channels):
    """(input channels x kernel, output channels, output frames per latent frame) of the graph."""
    rate, strides = (1, synthetic.SYNTHESIS_STRIDES) if synthesis else (HOP, synthetic.ANALYSIS_STRIDES)
    for i in range(30):
        first, kernel, last = synthetic.dac_shape(synthesis, channels, i)
        stage, within = divmod(i - 1, 7)
        if synthesis and 1 <= i <= 28 and within == 0:
            rate *= strides[stage]
            yield last * (kernel // strides[stage]), first, rate, first * kernel * last
            continue
        if not synthesis and 1 <= i <= 28 and within == 6:
            rate //= strides[stage]
        yield first * kernel, last, rate, first * kernel * last


def _codec_work(synthesis, case, frames):
    parts = list(_convolutions(synthesis, case["channels"]))
    rvq = case["books"] * (8192 * 2 + 1024)
    flops = sum(2 * taps * out * rate for taps, out, rate, _ in parts) + case["books"] * 2 * 8 * 1024
    data = 4 * HOP * case["channels"] + 2 * case["books"]
    return {"bytes": 4 * sum(p[3] for p in parts) + 4 * rvq + frames * data, "flops": frames * flops}


def _model_work(g, frames, books, batch):
    temporal = sum(k * n for k, n in (g.projection_shape(p) for p in range(4))) * g.temporal_layers
    codebook = sum(k * n for k, n in (g.projection_shape(p) for p in range(4))) * g.codebook_layers
    per_token = codebook + 2 * g.latent * g.width + g.width * g.alphabet
    length = min(g.context, -(-frames // batch))
    attention = 4 * g.width * (g.temporal_layers * (length + 1) / 2 + books * g.codebook_layers * (books + 1) / 2)
    flops = frames * (2 * temporal + attention + books * 2 * per_token)
    weights = sum(_linear_bytes(*g.projection_shape(p)) for p in range(g.projection_count))
    tokens = frames * books
    return {"bytes": weights + tokens * 2 * g.latent + tokens * 2 + tokens * 10 // 8, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["rows"], case["K"], case["N"]
        return {"bytes": 2 * m * (k + n) + _linear_bytes(k, n), "flops": 2 * m * k * n}
    if kind == "mlp":
        g, m = GEOMETRIES[case["geometry"]], case["rows"]
        return {"bytes": 4 * m * g.width + _linear_bytes(g.width, g.ffn) + _linear_bytes(g.ffn, g.width),
                "flops": 4 * m * g.width * g.ffn}
    if kind == "head":
        g, m = GEOMETRIES[case["geometry"]], case["rows"]
        return {"bytes": 2 * m * (g.width + 2 * g.alphabet) + _linear_bytes(g.width, g.alphabet),
                "flops": 2 * m * g.width * g.alphabet}
    if kind == "attention_step":
        n, t, w = case["sequences"], case["time"], case["heads"] * case["head_width"]
        return {"bytes": 4 * n * t * w + 4 * n * w, "flops": 4 * n * t * w}
    if kind == "attention_causal":
        lengths, w = _lengths(case), case["heads"] * case["head_width"]
        return {"bytes": 8 * sum(lengths) * w, "flops": sum(2 * w * t * (t + 1) for t in lengths)}
    if kind in ("synthesis", "analysis"):
        return _codec_work(kind == "synthesis", case, case["frames"])
    frames = case["frames"] if "frames" in case else -(-case["samples"] // HOP)
    model = _model_work(_geometry(case), frames, case["books"], case["batch"])
    if kind in ("audio_encode", "audio_decode"):
        codec = _codec_work(kind == "audio_decode", case, frames)
        return {key: model[key] + codec[key] for key in model}
    return model


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------- 64-bit results

def _exact_quantized(x):
    """BF8L activations: per 256 values a scale (in BF16) and whole numbers up to 127."""
    blocks = x.reshape(x.shape[0], -1, 256)
    scale = (blocks.abs().amax(-1, keepdim=True).float() / 127).clamp_min(1e-35).to(torch.bfloat16).float()
    whole = torch.round(blocks.float() * (1 / scale)).clamp(-127, 127).double()
    return whole * scale.double()


def _exact_linear(x, weights):
    values, scales, bias = (torch.from_numpy(a).cuda().double() for a in weights)
    n, k = values.shape
    dense = (values.reshape(n, k // 256, 256) * scales.t()[:, :, None]).reshape(n, k)
    return _exact_quantized(x).reshape(x.shape[0], k) @ dense.t() + bias


def _exact_norm(x, gain, bias):
    centred = x - x.mean(-1, keepdim=True)
    return centred / torch.sqrt(centred.square().mean(-1, keepdim=True) + 1e-5) * gain + bias


def _exact_rotary(x, rotations):
    """x [time][heads][head_width], pairs of neighbours turned by (cos, sin)."""
    table = _numbers(rotations[:x.shape[0]]).double()[:, None, :]
    cos, sin = table[..., 0::2], table[..., 1::2]
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).reshape(x.shape)


def _exact_attention(query, keys, values, mask=None):
    """query [q][heads][w], keys and values [t][heads][w]."""
    scores = torch.matmul(query.transpose(0, 1), keys.permute(1, 2, 0).contiguous()) / math.sqrt(query.shape[-1])
    if mask is not None:
        scores = scores.masked_fill(mask, -math.inf)
    return torch.matmul(torch.softmax(scores, -1), values.transpose(0, 1).contiguous()).transpose(0, 1)


def _exact_fold(columns, gain):
    """Weight norm: each row scaled to its gain."""
    return columns / columns.square().sum(-1, keepdim=True).sqrt() * gain[:, None]


def _exact_convolution_weights(conv):
    first, kernel, last = conv.dims
    values = torch.from_numpy(conv.values).cuda().double().reshape(last, kernel, first)
    if conv.bf8:
        scales = torch.from_numpy(synthetic.bf16_float(conv.scales)).cuda().double()[:, :, :kernel]
        values = values * scales.transpose(1, 2).repeat_interleave(32, -1)
    gain = torch.from_numpy(conv.gain).cuda().double()
    return _exact_fold(values.reshape(last, -1), gain).reshape(last, kernel, first)


def _exact_convolution(x, conv, stride, dilation):
    """x [channels][frames]."""
    w, bias = _exact_convolution_weights(conv), torch.from_numpy(conv.bias).cuda().double()[:, None]
    kernel, frames = w.shape[1], x.shape[1]
    if conv.transposed:
        full = x.new_zeros(w.shape[2], (frames - 1) * stride + kernel)
        for tap in range(kernel):
            full[:, tap:tap + (frames - 1) * stride + 1:stride] += w[:, tap, :].t().contiguous() @ x
        padding = (stride + 1) // 2
        return full[:, padding:full.shape[1] - padding] + bias
    padding = (kernel - 1) * dilation // 2
    padded = torch.nn.functional.pad(x, (padding, padding))
    out = bias.expand(-1, frames).clone()
    for tap in range(kernel):
        out += w[:, tap, :].contiguous() @ padded[:, tap * dilation:tap * dilation + frames]
    return out


def _exact_snake(x, alpha):
    a = torch.from_numpy(alpha).cuda().double()[:, None]
    return x + torch.sin(a * x).square() / (a + 1e-9)


def _exact_synthesis(case, seed):
    dac = synthetic.random_dac(case["channels"], 12 if case["channels"] == 2 else 9, seed)
    tokens = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda().reshape(case["frames"], case["books"])
    x = 0
    for b in range(case["books"]):
        codebook, out_v, out_g, out_bias = (torch.from_numpy(np.asarray(a[b])).cuda().double() for a in (
            dac.codebook, dac.out_v, dac.out_g, dac.out_bias))
        x = x + _exact_fold(out_v, out_g) @ codebook[tokens[:, b]].t() + out_bias[:, None]
    convs, alphas = dac.synthesis, dac.synthesis_alpha
    x = _exact_convolution(x, convs[0], 1, 1)
    for stage, stride in enumerate(synthetic.SYNTHESIS_STRIDES):
        at = 7 * stage
        x = _exact_convolution(_exact_snake(x, alphas[at]), convs[at + 1], stride, 1)
        for unit, dilation in enumerate((1, 3, 9)):
            y = _exact_convolution(_exact_snake(x, alphas[at + 1 + 2 * unit]), convs[at + 2 + 2 * unit], 1, dilation)
            y = _exact_convolution(_exact_snake(y, alphas[at + 2 + 2 * unit]), convs[at + 3 + 2 * unit], 1, 1)
            x = x + y
    x = _exact_convolution(_exact_snake(x, alphas[28]), convs[29], 1, 1)
    return x.t().contiguous().reshape(-1).cpu().numpy()


def exact(case, seed):
    """Operators and codec synthesis in 64 bits, quantised to BF8L where the
    operator quantises. Streams have no such value (every bit of each
    probability is the format's own); a decoded stream's tokens are the encoded ones."""
    kind = case["kind"]
    if kind in ("linear", "mlp", "head"):
        weights = _weights(case, seed)
        x = _numbers(_normal(seed, 1, (case["rows"], weights[0][0].shape[1]))).double()
        if kind == "linear":
            return _exact_linear(x, weights[0])
        gain, bias = (_numbers(a).double() for a in _norm(case, seed))
        hidden = _exact_linear(_exact_norm(x, gain, bias), weights[0])
        if kind == "head":
            return hidden, torch.softmax(hidden, -1)
        active = torch.nn.functional.gelu(hidden, approximate="tanh")
        return x + _exact_linear(active, weights[1])
    if kind == "attention_step":
        n, t, heads, hw = case["sequences"], case["time"], case["heads"], case["head_width"]
        q, k, v = (_numbers(_normal(seed, salt, shape)).double() for salt, shape in (
            (1, (n, 1, heads, hw)), (2, (n, t, heads, hw)), (3, (n, t, heads, hw))))
        return torch.stack([_exact_attention(q[i], k[i], v[i]) for i in range(n)]).reshape(n, heads * hw)
    if kind == "attention_causal":
        heads, hw, rotations = case["heads"], case["head_width"], _rotations(case["head_width"], 1024)
        lengths, outputs = _lengths(case), []
        qkv = _numbers(_normal(seed, 1, (sum(lengths), 3 * heads * hw))).double()
        for rows in torch.split(qkv, lengths):
            t = rows.shape[0]
            q, k, v = rows.reshape(t, 3, heads, hw).unbind(1)
            mask = torch.ones(t, t, dtype=torch.bool, device="cuda").triu(1)
            out = _exact_attention(_exact_rotary(q, rotations), _exact_rotary(k, rotations), v, mask)
            outputs.append(out.reshape(t, heads * hw))
        return torch.cat(outputs)
    if kind == "synthesis":
        return _exact_synthesis(case, seed)
    if kind == "model_decode":
        return _tokens(case, seed)
    return None
