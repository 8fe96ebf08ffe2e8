"""The measured workloads: what a speech-to-text program has this library do,
through the Python binding's public calls, over the sizes that it meets.

A program opens one context, binds its model's matrices, and then, for each
clip, runs the convolution front end, the audio tower's layers, the prompt
prefill and the greedy steps; a server runs the steps for several sequences at
once. The listed cases are the single products of those stages (one token, a
few sequences, a prompt's rows; every weight format), the attentions, the two
audio stages, and two whole calls. Matrix shapes are those of the 0.6B and
1.7B configurations in this repository's benchmark and tests; weights and
inputs are synthetic, made from the seed.
"""
import math

import numpy as np
import torch

import qwenscriber_amd as qa

DEVICE = "cuda"
FORMATS = {"q4": qa.FORMAT_Q4, "q5": qa.FORMAT_Q5, "q8": qa.FORMAT_Q8, "f16": qa.FORMAT_F16, "f32": qa.FORMAT_F32}
BIAS = {"q4": 8, "q5": 16, "q8": 128}
WEIGHT_BYTES = {"q4": 34 / 64, "q5": 42 / 64, "q8": 66 / 64, "f16": 2.0, "f32": 4.0}
WEIGHT_SCALE = 0.02
EPS = 1e-6
THETA = 1e6
VOCAB = 151936
AUDIO_PAD = 151676
LAYERS = 28
# hidden, ffn of the two text decoders (16 query heads over 8 key/value heads
# of 128), and d_model, ffn, heads of the audio tower.
DECODERS = {"0.6b": (1024, 3072), "1.7b": (2048, 6144)}
HEADS, KV_HEADS, HEAD_DIM = 16, 8, 128
D_MODEL, AUDIO_FFN, AUDIO_HEADS, WINDOW = 896, 3584, 14, 104
MEL_BINS, N_WINDOW, CHANNELS = 128, 50, 480
# The products of a 0.6B and a 1.7B model, rows x columns.
PRODUCTS = [(4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072), (4096, 2048), (2048, 2048), (12288, 2048),
            (2048, 6144), (896, 896), (3584, 896), (896, 3584), (1024, 896), (896, 7680)]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
_context = None


def context():
    """The program's one context: a device and a stream."""
    global _context
    if _context is None:
        _context = qa.Context(0)
    return _context


class Inputs:
    """Values in a fixed order from one seed."""

    def __init__(self, seed):
        self.generator = torch.Generator(device=DEVICE)
        self.generator.manual_seed(1000003 * int(seed) + 17)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.generator, device=DEVICE, dtype=torch.float32) * scale

    def integers(self, high, count):
        return torch.randint(0, high, (count,), generator=self.generator, device=DEVICE, dtype=torch.int64)

    def weights(self, fmt, rows, cols, scale=WEIGHT_SCALE):
        return Weights(fmt, self.normal(rows, cols, scale=scale))


class Weights:
    """A matrix in one of the storage formats: groups of 64 values with an f16
    scale and biased codes, or f16 / f32 elements."""

    def __init__(self, fmt, values):
        self.fmt = fmt
        self.rows, self.cols = values.shape
        if fmt in BIAS:
            self.codes, self.scale = quantize(values, BIAS[fmt])
        else:
            self.elements = values.half() if fmt == "f16" else values

    def planes(self):
        """(scale plane, data plane) as byte tensors; no scale plane for elements."""
        if self.fmt not in BIAS:
            return None, self.elements.contiguous().view(torch.uint8)
        return self.scale.contiguous().view(torch.uint8), pack(self.fmt, self.codes)

    def exact(self):
        if self.fmt not in BIAS:
            return self.elements.double()
        return dequantized(self.codes, self.scale)

    def exact_rows(self, at):
        if self.fmt not in BIAS:
            return self.elements[at].double()
        return dequantized(self.codes[at], self.scale[at])

    def times(self, x):
        """x [tokens][cols] in f64 times the matrix, a stretch of rows at a time."""
        step = max(1, (1 << 27) // self.cols)
        parts = []
        for r in range(0, self.rows, step):
            at = slice(r, min(self.rows, r + step))
            parts.append(x @ self.exact_rows(at).t().contiguous())
        return torch.cat(parts, dim=1)


def quantize(values, bias):
    """Codes (int16, centred on zero) and f16 scales of groups of 64."""
    groups = values.reshape(values.shape[0], -1, 64)
    scale = (groups.abs().amax(dim=2) / bias).half()
    stored = scale.to(values.dtype).unsqueeze(2)
    ratio = torch.where(stored == 0, torch.zeros_like(groups), groups / stored)
    codes = torch.where(ratio >= 0, torch.floor(ratio + 0.5), torch.ceil(ratio - 0.5)).clamp_(-bias, bias - 1)
    return codes.to(torch.int16), scale


def dequantized(codes, scale):
    return (codes.double() * scale.double().unsqueeze(2)).reshape(codes.shape[0], -1)


def pack(fmt, codes):
    """The data plane: q8 bytes; q4 / q5 nibbles with the even column low, and
    for q5 the fifth bits after each group's nibbles."""
    u = (codes + BIAS[fmt]).to(torch.uint8)
    if fmt == "q8":
        return u.contiguous()
    low = u & 15
    nibbles = low[..., 0::2] | (low[..., 1::2] << 4)
    if fmt == "q4":
        return nibbles.contiguous()
    fifth = (u >> 4).reshape(*u.shape[:2], 8, 8)
    bits = torch.zeros_like(fifth[..., 0])
    for j in range(8):
        bits |= fifth[..., j] << j
    return torch.cat([nibbles, bits], dim=2).contiguous()


class State:
    """What a program holds between calls: device tensors, matrix handles and
    perhaps a decoder."""

    def __init__(self, case):
        self.case = case
        self.ctx = context()
        self.handles = []
        self.keep = []
        self.decoder = None

    def matrix(self, weights):
        scales, data = weights.planes()
        torch.cuda.synchronize()
        self.keep += [scales, data]
        handle = self.ctx.matrix_wrap(FORMATS[weights.fmt], weights.rows, weights.cols,
                                      0 if scales is None else scales.data_ptr(), data.data_ptr())
        self.handles.append(handle)
        return handle

    def __del__(self):
        if getattr(self, "ctx", None) is None or not self.ctx.handle:
            return
        self.ctx.sync()
        if self.decoder is not None:
            self.decoder.close()
        for handle in self.handles:
            self.ctx.matrix_release(handle)


def empty(*shape):
    return torch.empty(*shape, device=DEVICE, dtype=torch.float32)


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: two sequences through the 0.6B down projection,
        # where the launches and first bytes count.
        {"name": "linear_q8_down_t2", "kind": "linear", "format": "q8", "rows": 1024, "cols": 3072, "tokens": 2},
        # The largest one-token product, once per decoded token: the 1.7B
        # vocabulary head, a stream of its weights.
        {"name": "linear_q4_head_t1", "kind": "linear", "format": "q4", "rows": VOCAB, "cols": 2048, "tokens": 1},
        # A server's step for 16 sequences: the widest layer product.
        {"name": "linear_q4_gate_up_t16", "kind": "linear", "format": "q4", "rows": 12288, "cols": 2048, "tokens": 16},
        # A 30 s prompt's rows through a layer product (f32 activations).
        {"name": "linear_q8_prompt_t402", "kind": "linear", "format": "q8", "rows": 2048, "cols": 6144, "tokens": 402},
        # An unquantized model, an odd number of rows.
        {"name": "linear_f16_t37", "kind": "linear", "format": "f16", "rows": 4096, "cols": 2048, "tokens": 37},
        # bf16 activations, two minutes of audio steps.
        {"name": "gemm_bf16_q4_t1500", "kind": "gemm", "format": "q4", "rows": 6144, "cols": 2048, "tokens": 1500},
        # A server's decode attention: 16 sequences of 4096 cached positions.
        {"name": "attention_q8_b16", "kind": "attention", "cache": "q8", "cached": 4096, "batch": 16},
        # One sequence over the default f32 cache, at an odd position.
        {"name": "attention_f32_b1", "kind": "attention", "cache": "f32", "cached": 3001, "batch": 1},
        # One layer of the audio tower over a 30 s clip.
        {"name": "audio_layer_q8", "kind": "audio_layer", "format": "q8", "steps": 390},
        # The convolution front end over a 30 s clip.
        {"name": "frontend_30s", "kind": "frontend", "format": "q8", "frames": 3000},
        # The prompt of a 30 s clip through a whole decoder, to its logits.
        {"name": "prefill_1.7b_402", "kind": "prefill", "model": "1.7b", "format": "q4", "cache": "q8", "count": 402,
         "audio": 390, "first": 0},
        # Four decode steps of a single transcription after such a prompt.
        {"name": "steps_0.6b_b1", "kind": "steps", "model": "0.6b", "format": "q8", "cache": "q8", "first": 450,
         "steps": 4, "batch": 1},
    ]


def log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "gemm", "attention", "audio_layer", "frontend", "prefill", "steps"])
    quantized = rng.choice(["q4", "q5", "q8"])
    if kind == "linear":
        rows, cols = rng.choice(PRODUCTS)
        tokens = log_int(rng, 1, 512)
        if rng.random() < 0.15:
            rows, cols, tokens = VOCAB, rng.choice([1024, 2048]), log_int(rng, 1, 16)
        elif rng.random() < 0.25:  # shapes of no listed model
            rows, cols = log_int(rng, 65, 8191), 64 * log_int(rng, 2, 96)
        elif tokens == 1:  # a product that outlasts its launch
            rows, cols = VOCAB, rng.choice([1024, 2048])
        fmt = rng.choice(["q4", "q4", "q5", "q8", "q8", "f16", "f32"])
        if fmt == "q5" and cols > 6144:  # one-token q5 rows end there
            fmt = "q8"
        return {"kind": kind, "format": fmt, "rows": rows, "cols": cols, "tokens": tokens}
    if kind == "gemm":
        rows, cols = rng.choice(PRODUCTS)
        return {"kind": kind, "format": quantized, "rows": rows, "cols": cols, "tokens": log_int(rng, 17, 2048)}
    if kind == "attention":
        return {"kind": kind, "cache": rng.choice(["q8", "f32"]), "cached": log_int(rng, 33, 8192),
                "batch": log_int(rng, 1, 16)}
    if kind == "audio_layer":
        return {"kind": kind, "format": quantized, "steps": log_int(rng, 13, 780)}
    if kind == "frontend":
        return {"kind": kind, "format": quantized, "frames": log_int(rng, 90, 3000)}
    model = rng.choice(sorted(DECODERS))
    cache = rng.choice(["q8", "q8", "f32"])
    if kind == "prefill":
        count = log_int(rng, 9, 512)
        return {"kind": kind, "model": model, "format": rng.choice(["q4", "q5", "q8"]), "cache": cache,
                "count": count, "audio": int(count * rng.uniform(0.5, 0.97)), "first": 0}
    return {"kind": kind, "model": model, "format": quantized, "cache": cache, "first": log_int(rng, 40, 2048),
            "steps": 2, "batch": rng.choice([1, 1, 2, 4, 7])}


# ---------------------------------------------------------------------------
# Single products
# ---------------------------------------------------------------------------
def linear_inputs(case, seed):
    i = Inputs(seed)
    w = i.weights(case["format"], case["rows"], case["cols"])
    return w, i.normal(case["tokens"], case["cols"])


def prepare_linear(case, seed):
    w, x = linear_inputs(case, seed)
    s = State(case)
    s.weights = s.matrix(w)
    s.x = x.bfloat16() if case["kind"] == "gemm" else x
    s.out = empty(case["tokens"], case["rows"])
    return s


def run_linear(s):
    c = s.case
    call = s.ctx.linear_bf16 if c["kind"] == "gemm" else s.ctx.linear
    call(s.weights, s.x.data_ptr(), c["cols"], c["tokens"], s.out.data_ptr())
    return s.out


def exact_linear(case, seed):
    w, x = linear_inputs(case, seed)
    return w.times((x.bfloat16() if case["kind"] == "gemm" else x).double())


def work_linear(case):
    n, k, m = case["rows"], case["cols"], case["tokens"]
    x_bytes = 2 if case["kind"] == "gemm" else 4
    return {"bytes": n * k * WEIGHT_BYTES[case["format"]] + m * (x_bytes * k + 4 * n), "flops": 2 * m * n * k}


# ---------------------------------------------------------------------------
# Decode attention
# ---------------------------------------------------------------------------
def attention_inputs(case, seed):
    i = Inputs(seed)
    width = KV_HEADS * HEAD_DIM
    q = i.normal(case["batch"], HEADS * HEAD_DIM)
    planes = [i.normal(case["batch"] * case["cached"], width) for _ in range(2)]
    return q, [Weights("q8", p) if case["cache"] == "q8" else p for p in planes]


def prepare_attention(case, seed):
    s = State(case)
    s.q, planes = attention_inputs(case, seed)
    if case["cache"] == "q8":
        s.planes = [p.contiguous() for w in planes for p in w.planes()]
    else:
        s.planes = planes
    s.out = empty(case["batch"], HEADS * HEAD_DIM)
    return s


def run_attention(s):
    c = s.case
    n, width = c["cached"], KV_HEADS * HEAD_DIM
    p = [t.data_ptr() for t in s.planes]
    if c["cache"] == "q8":
        s.ctx.decode_attention_q8(s.out.data_ptr(), s.q.data_ptr(), p[0], p[1], p[2], p[3], n, HEADS, KV_HEADS,
                                  HEAD_DIM, c["batch"], n * width // 32, n * width)
    else:
        s.ctx.decode_attention_f32(s.out.data_ptr(), s.q.data_ptr(), p[0], p[1], n, HEADS, KV_HEADS, HEAD_DIM,
                                   c["batch"], n * width * 4)
    return s.out


def attend(q, keys, values, mask=None):
    """q [rows][heads][d], keys / values [positions][kv_heads][d] in f64."""
    ratio = q.shape[1] // keys.shape[1]
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        scores = q[:, h].contiguous() @ keys[:, h // ratio].t().contiguous() / math.sqrt(q.shape[2])
        if mask is not None:
            scores = scores.masked_fill(mask, -math.inf)
        out[:, h] = torch.softmax(scores, dim=1) @ values[:, h // ratio].contiguous()
    return out


def exact_attention(case, seed):
    q, planes = attention_inputs(case, seed)
    keys, values = [(p.exact() if case["cache"] == "q8" else p.double()).reshape(case["batch"], -1, KV_HEADS, HEAD_DIM)
                    for p in planes]
    q = q.double().reshape(case["batch"], 1, HEADS, HEAD_DIM)
    return torch.stack([attend(q[b], keys[b], values[b]).reshape(-1) for b in range(case["batch"])])


def work_attention(case):
    row = KV_HEADS * HEAD_DIM * (66 / 64 if case["cache"] == "q8" else 4)
    positions = case["batch"] * case["cached"]
    return {"bytes": 2 * positions * row + 8 * case["batch"] * HEADS * HEAD_DIM,
            "flops": 4 * positions * HEADS * HEAD_DIM}


# ---------------------------------------------------------------------------
# Audio tower layer
# ---------------------------------------------------------------------------
AUDIO_MATRICES = {"q": (D_MODEL, D_MODEL), "k": (D_MODEL, D_MODEL), "v": (D_MODEL, D_MODEL), "o": (D_MODEL, D_MODEL),
                  "ffn_in": (AUDIO_FFN, D_MODEL), "ffn_out": (D_MODEL, AUDIO_FFN)}


def audio_inputs(case, seed):
    i = Inputs(seed)
    matrices = {name: i.weights(case["format"], *shape) for name, shape in AUDIO_MATRICES.items()}
    vectors = {}
    for name in qa.AudioLayerWeights.VECTORS:
        v = i.normal(AUDIO_FFN if name == "ffn_in_bias" else D_MODEL, scale=0.1)
        vectors[name] = 1.0 + v if name.endswith("norm_weight") else v
    return matrices, vectors, i.normal(case["steps"], D_MODEL)


def prepare_audio_layer(case, seed):
    s = State(case)
    matrices, s.vectors, s.encoder = audio_inputs(case, seed)
    s.weights = qa.AudioLayerWeights()
    for name, w in matrices.items():
        setattr(s.weights, name, s.matrix(w))
    for name, v in s.vectors.items():
        setattr(s.weights, name, v.data_ptr())
    return s


def run_audio_layer(s):
    # The residual stream is updated in place, as the tower's layers do.
    s.ctx.audio_layer(s.weights, s.encoder.data_ptr(), s.case["steps"], D_MODEL, AUDIO_HEADS, AUDIO_FFN, WINDOW, 1e-5)
    return s.encoder


def gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def exact_audio_layer(case, seed):
    matrices, vectors, encoder = audio_inputs(case, seed)
    v = {name: t.double() for name, t in vectors.items()}
    x = encoder.double()
    norm = torch.nn.functional.layer_norm
    head = (-1, AUDIO_HEADS, D_MODEL // AUDIO_HEADS)
    y = norm(x, (D_MODEL,), v["attention_norm_weight"], v["attention_norm_bias"], 1e-5)
    q, k, val = [(matrices[n].times(y) + v[n + "_bias"]).reshape(head) for n in ("q", "k", "v")]
    parts = [attend(q[a:a + WINDOW], k[a:a + WINDOW], val[a:a + WINDOW]) for a in range(0, case["steps"], WINDOW)]
    x = x + (matrices["o"].times(torch.cat(parts).reshape(-1, D_MODEL)) + v["o_bias"])
    y = norm(x, (D_MODEL,), v["final_norm_weight"], v["final_norm_bias"], 1e-5)
    y = gelu(matrices["ffn_in"].times(y) + v["ffn_in_bias"])
    return x + (matrices["ffn_out"].times(y) + v["ffn_out_bias"])


def work_audio_layer(case):
    t = case["steps"]
    values = sum(r * c for r, c in AUDIO_MATRICES.values())
    pairs = sum(min(WINDOW, t - a) ** 2 for a in range(0, t, WINDOW))
    return {"bytes": values * WEIGHT_BYTES[case["format"]] + 8 * t * D_MODEL,
            "flops": 2 * t * values + 4 * pairs * D_MODEL}


# ---------------------------------------------------------------------------
# Audio convolution front end
# ---------------------------------------------------------------------------
def halved(n):
    return (n - 1) // 2 + 1


def thrice_halved(n):
    return halved(halved(halved(n))) if n else 0


def encoder_rows(frames):
    chunk = 2 * N_WINDOW
    return frames // chunk * thrice_halved(chunk) + thrice_halved(frames % chunk)


def frontend_inputs(case, seed):
    i = Inputs(seed)
    convolutions = []
    for cin in (1, CHANNELS, CHANNELS):
        w = i.normal(CHANNELS, cin, 3, 3, scale=1.0 / math.sqrt(9 * cin)).half()
        convolutions.append((w, i.normal(CHANNELS, scale=0.1)))
    out = i.weights(case["format"], D_MODEL, CHANNELS * thrice_halved(MEL_BINS))
    return convolutions, out, i.normal(MEL_BINS, case["frames"])


def prepare_frontend(case, seed):
    s = State(case)
    s.convolutions, out, s.mel = frontend_inputs(case, seed)
    s.weights = qa.AudioFrontendWeights()
    for j, (w, b) in enumerate(s.convolutions):
        setattr(s.weights, f"conv{j + 1}_weight", w.data_ptr())
        setattr(s.weights, f"conv{j + 1}_bias", b.data_ptr())
    s.weights.conv_out = s.matrix(out)
    s.out = empty(encoder_rows(case["frames"]), D_MODEL)
    return s


def run_frontend(s):
    s.ctx.audio_frontend(s.weights, s.mel.data_ptr(), MEL_BINS, s.case["frames"], N_WINDOW, CHANNELS, D_MODEL,
                         s.out.data_ptr(), s.out.shape[0])
    return s.out


def exact_frontend(case, seed):
    convolutions, out, mel = frontend_inputs(case, seed)
    frames, chunk = case["frames"], 2 * N_WINDOW
    chunks = -(-frames // chunk)
    padded = torch.zeros(MEL_BINS, chunks * chunk, device=DEVICE, dtype=torch.float64)
    padded[:, :frames] = mel.double()
    x = padded.reshape(MEL_BINS, chunks, chunk).permute(1, 0, 2).unsqueeze(1).contiguous()
    for w, b in convolutions:
        h, width = halved(x.shape[2]), halved(x.shape[3])
        w64 = w.double().reshape(CHANNELS, -1)
        images = []
        for image in x:
            columns = torch.nn.functional.unfold(image.unsqueeze(0), 3, padding=1, stride=2)[0]
            images.append((w64 @ columns + b.double().unsqueeze(1)).reshape(CHANNELS, h, width))
        x = gelu(torch.stack(images))
    rows = x.permute(0, 3, 1, 2).reshape(chunks * x.shape[3], -1)[:encoder_rows(frames)].contiguous()
    half = D_MODEL // 2
    inverse = torch.exp(torch.arange(half, device=DEVICE, dtype=torch.float64) * (-math.log(10000.0) / (half - 1)))
    step = torch.arange(rows.shape[0], device=DEVICE, dtype=torch.float64) % thrice_halved(chunk)
    angle = step.unsqueeze(1) * inverse
    return out.times(rows) + torch.cat([torch.sin(angle), torch.cos(angle)], dim=1)


def work_frontend(case):
    chunks = -(-case["frames"] // (2 * N_WINDOW))
    h, width, macs, values = MEL_BINS, 2 * N_WINDOW, 0, 0
    for cin in (1, CHANNELS, CHANNELS):
        h, width = halved(h), halved(width)
        macs += chunks * CHANNELS * h * width * cin * 9
        values += CHANNELS * cin * 9
    rows, features = encoder_rows(case["frames"]), CHANNELS * thrice_halved(MEL_BINS)
    return {"bytes": 2 * values + D_MODEL * features * WEIGHT_BYTES[case["format"]] +
            4 * MEL_BINS * case["frames"] + 4 * rows * D_MODEL,
            "flops": 2 * (macs + rows * D_MODEL * features)}


# ---------------------------------------------------------------------------
# Whole decoder calls
# ---------------------------------------------------------------------------
KINDS = {"q": qa.T_Q, "k": qa.T_K, "v": qa.T_V, "o": qa.T_O, "gate": qa.T_GATE, "up": qa.T_UP, "down": qa.T_DOWN}


def layer_shapes(model):
    hidden, ffn = DECODERS[model]
    wide, kv = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    return {"q": (wide, hidden), "k": (kv, hidden), "v": (kv, hidden), "o": (hidden, wide), "gate": (ffn, hidden),
            "up": (ffn, hidden), "down": (hidden, ffn)}


def model_parts(case, seed):
    """(name, layer, Weights or norm vector) of a synthetic model, in order."""
    hidden, _ = DECODERS[case["model"]]
    i = Inputs(seed)
    yield "embed", 0, i.weights(case["format"], VOCAB, hidden)
    for layer in range(LAYERS):
        for name, shape in layer_shapes(case["model"]).items():
            yield name, layer, i.weights(case["format"], *shape)
        for name, width in (("attn_norm", hidden), ("q_norm", HEAD_DIM), ("k_norm", HEAD_DIM), ("ffn_norm", hidden)):
            yield name, layer, 1.0 + i.normal(width, scale=0.1)
    yield "final_norm", 0, 1.0 + i.normal(hidden, scale=0.1)
    yield "lm_head", 0, i.weights(case["format"], VOCAB, hidden)


NORMS = {"attn_norm": qa.T_ATTN_NORM, "q_norm": qa.T_Q_NORM, "k_norm": qa.T_K_NORM, "ffn_norm": qa.T_FFN_NORM,
         "final_norm": qa.T_FINAL_NORM}


def model_decoder(s, case, seed, batch, max_positions):
    hidden, ffn = DECODERS[case["model"]]
    ctx = s.ctx
    s.decoder = qa.Decoder(ctx, batch=batch, cache_format=qa.CACHE_Q8 if case["cache"] == "q8" else qa.CACHE_F32,
                           hidden=hidden, layers=LAYERS, heads=HEADS, kv_heads=KV_HEADS, head_dim=HEAD_DIM, ffn=ffn,
                           vocab=VOCAB, max_positions=max_positions, eps=EPS, theta=THETA)
    for name, layer, part in model_parts(case, seed):
        if name in NORMS:
            s.decoder.set_vector(NORMS[name], layer, part.cpu().numpy())
            continue
        scales, data = part.planes()
        torch.cuda.synchronize()
        handle = ctx.matrix_wrap(FORMATS[part.fmt], part.rows, part.cols,
                                 0 if scales is None else scales.data_ptr(), data.data_ptr())
        kind = {"embed": qa.T_EMBED, "lm_head": qa.T_LM_HEAD}.get(name)
        s.decoder.set_matrix(KINDS[name] if kind is None else kind, layer, handle)
        ctx.sync()  # the decoder has its copy: these planes may go
        ctx.matrix_release(handle)


def prompt_inputs(case, seed):
    hidden, _ = DECODERS[case["model"]]
    i = Inputs(seed + 7919)
    tokens = i.integers(AUDIO_PAD, case["count"]).cpu().numpy().astype(np.uint32)
    start = (case["count"] - case["audio"]) // 2
    tokens[start:start + case["audio"]] = AUDIO_PAD
    return tokens, i.normal(max(1, case["audio"]), hidden, scale=WEIGHT_SCALE)


def prepare_prefill(case, seed):
    s = State(case)
    s.tokens, s.rows = prompt_inputs(case, seed)
    model_decoder(s, case, seed, 1, 1024)
    return s


def run_prefill(s):
    c = s.case
    s.decoder.set_position(0, c["first"])
    s.decoder.prefill(0, s.tokens, AUDIO_PAD, s.rows.data_ptr(), c["audio"])
    return s.decoder.logits(0)


def cache_inputs(case, seed):
    """Per sequence and layer, the cached keys and values: (Weights or f32) pairs."""
    i = Inputs(seed + 104729)
    width = KV_HEADS * HEAD_DIM
    for b in range(case["batch"]):
        for layer in range(LAYERS):
            pair = [i.normal(case["first"], width) for _ in range(2)]
            yield b, layer, [Weights("q8", p) if case["cache"] == "q8" else p for p in pair]


def step_tokens(case, seed):
    return Inputs(seed + 15485863).integers(AUDIO_PAD, case["steps"] * case["batch"]).cpu().numpy().astype(
        np.uint32).reshape(case["steps"], case["batch"])


def prepare_steps(case, seed):
    s = State(case)
    s.tokens = step_tokens(case, seed)
    model_decoder(s, case, seed, case["batch"], case["first"] + case["steps"] + 64)

    def put(address, tensor):
        host = tensor.cpu().contiguous().numpy().view(np.uint8).reshape(-1)
        s.ctx._check(s.ctx.lib.qwh_upload(s.ctx.handle, address, host.ctypes.data, host.nbytes))

    for b, layer, pair in cache_inputs(case, seed):
        planes = s.decoder.cache_planes(b, layer)
        for j, part in enumerate(pair):
            if case["cache"] == "q8":
                scales, data = part.planes()
                put(planes[2 * j], scales)
                put(planes[2 * j + 1], data)
            else:
                put(planes[2 * j + 1], part)
    return s


def run_steps(s):
    c = s.case
    for b in range(c["batch"]):
        s.decoder.set_position(b, c["first"])
    for k in range(c["steps"]):
        s.decoder.forward(s.tokens[k], k + 1 == c["steps"])
    return np.stack([s.decoder.logits(b) for b in range(c["batch"])])


def rms_norm(x, weight):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * weight.double()


def rotate(x, positions):
    """Rotary positions over [rows][heads][d], the angles in f32 as the model's tables have them."""
    half = HEAD_DIM // 2
    inverse = np.power(float(THETA), -2.0 * np.arange(half) / HEAD_DIM).astype(np.float32)
    angle = (positions.astype(np.float32)[:, None] * inverse[None, :]).astype(np.float32).astype(np.float64)
    cos, sin = [torch.from_numpy(f(angle)).to(DEVICE).unsqueeze(1) for f in (np.cos, np.sin)]
    low, high = x[..., :half], x[..., half:]
    return torch.cat([low * cos - high * sin, high * cos + low * sin], dim=-1)


def stored(rows, cache):
    """What a cache of this format gives back for the rows [n][kv_heads * d]."""
    return dequantized(*quantize(rows, 128)) if cache == "q8" else rows


def exact_layers(case, parts, x, positions, cached, sequences):
    """The decoder's layers in f64 over rows x. `cached(layer)` gives per
    sequence the earlier keys and values; sequences[r] is row r's sequence, its
    rows in order of position. `parts` is consumed up to the layers' end."""
    n = x.shape[0]
    for layer in range(LAYERS):
        w = {}
        for _ in range(11):
            name, _, part = next(parts)
            w[name] = part
        y = rms_norm(x, w["attn_norm"])
        q = rotate(rms_norm(w["q"].times(y).reshape(n, HEADS, HEAD_DIM), w["q_norm"]), positions)
        k = rotate(rms_norm(w["k"].times(y).reshape(n, KV_HEADS, HEAD_DIM), w["k_norm"]), positions)
        k, v = [stored(t.reshape(n, -1), case["cache"]).reshape(n, KV_HEADS, HEAD_DIM) for t in (k, w["v"].times(y))]
        out = torch.empty_like(q)
        for b in sorted(set(sequences)):
            rows = [r for r in range(n) if sequences[r] == b]
            before = cached(layer, b)
            keys, values = [torch.cat([p, t[rows]]) if p is not None else t[rows] for p, t in zip(before, (k, v))]
            base = keys.shape[0] - len(rows)
            at = torch.arange(keys.shape[0], device=DEVICE).unsqueeze(0)
            mask = at > base + torch.arange(len(rows), device=DEVICE).unsqueeze(1)
            out[rows] = attend(q[rows], keys, values, mask)
        x = x + w["o"].times(out.reshape(n, -1))
        y = rms_norm(x, w["ffn_norm"])
        gate = w["gate"].times(y)
        x = x + w["down"].times(gate / (1.0 + torch.exp(-gate)) * w["up"].times(y))
    return x


def exact_prefill(case, seed):
    tokens, rows = prompt_inputs(case, seed)
    parts = model_parts(case, seed)
    embed = next(parts)[2]
    x = embed.exact_rows(torch.from_numpy(np.minimum(tokens, VOCAB - 1).astype(np.int64)).to(DEVICE))
    pads = torch.from_numpy(tokens == AUDIO_PAD).to(DEVICE)
    x[pads] = rows[:case["audio"]].double()
    x = exact_layers(case, parts, x, np.arange(case["count"]), lambda layer, b: (None, None), [0] * case["count"])
    norm, head = next(parts)[2], next(parts)[2]
    return head.times(rms_norm(x[-1:], norm)).reshape(-1).cpu().numpy()


def exact_steps(case, seed):
    cache = {}
    for b, layer, pair in cache_inputs(case, seed):
        cache[layer, b] = [(p.exact() if case["cache"] == "q8" else p.double()).reshape(-1, KV_HEADS, HEAD_DIM)
                           for p in pair]
    tokens = step_tokens(case, seed)
    parts = model_parts(case, seed)
    embed = next(parts)[2]
    # All steps at once, each row seeing its sequence's rows up to its own.
    order = [(k, b) for b in range(case["batch"]) for k in range(case["steps"])]
    x = embed.exact_rows(torch.tensor([int(tokens[k, b]) for k, b in order], device=DEVICE))
    positions = np.array([case["first"] + k for k, _ in order])
    x = exact_layers(case, parts, x, positions, lambda layer, b: cache[layer, b], [b for _, b in order])
    norm, head = next(parts)[2], next(parts)[2]
    last = x[[r for r, (k, _) in enumerate(order) if k + 1 == case["steps"]]]
    return head.times(rms_norm(last, norm)).cpu().numpy()


def model_work(case, rows, cached_rows, pairs):
    """Weights once (each row's logits where wanted), the cache rows read and written, the products of `rows`."""
    hidden, _ = DECODERS[case["model"]]
    layer = LAYERS * sum(r * c for r, c in layer_shapes(case["model"]).values())
    row = 2 * KV_HEADS * HEAD_DIM * (66 / 64 if case["cache"] == "q8" else 4)
    return {"bytes": (layer + VOCAB * hidden) * WEIGHT_BYTES[case["format"]] + LAYERS * cached_rows * row,
            "flops": 2 * rows * layer + 2 * VOCAB * hidden + LAYERS * 4 * pairs * HEADS * HEAD_DIM}


def work_prefill(case):
    n = case["count"]
    return model_work(case, n, n, n * (n + 1) // 2)


def work_steps(case):
    # The steps follow one another: each streams the weights and the cache.
    rows = case["batch"] * case["steps"]
    one = model_work(case, case["batch"], case["batch"] * case["first"], case["batch"] * case["first"])
    return {"bytes": case["steps"] * one["bytes"] + 4 * case["batch"] * VOCAB, "flops": rows / case["batch"] * one["flops"]}


# ---------------------------------------------------------------------------
STAGES = {
    "linear": (prepare_linear, run_linear, exact_linear, work_linear),
    "gemm": (prepare_linear, run_linear, exact_linear, work_linear),
    "attention": (prepare_attention, run_attention, exact_attention, work_attention),
    "audio_layer": (prepare_audio_layer, run_audio_layer, exact_audio_layer, work_audio_layer),
    "frontend": (prepare_frontend, run_frontend, exact_frontend, work_frontend),
    "prefill": (prepare_prefill, run_prefill, exact_prefill, work_prefill),
    "steps": (prepare_steps, run_steps, exact_steps, work_steps),
}


def prepare(case, seed):
    s = STAGES[case["kind"]][0](case, seed)
    torch.cuda.synchronize()  # the library has a stream of its own
    return s


def run(state):
    return STAGES[state.case["kind"]][1](state)


def exact(case, seed):
    if case["kind"] in ("prefill", "steps") and case["cache"] == "q8":
        # The rounding of a new key or value to 8 bits is a step, not a sum:
        # a row a hair off the 64-bit one may round to another code, and the
        # distance from 64 bits then says which codes were near a tie.
        return None
    return STAGES[case["kind"]][2](case, seed)


def work(case):
    return STAGES[case["kind"]][3](case)


def tolerance(case):
    # About four times what the paths were seen to differ from 64 bits by, on
    # either side. Single layers and products: f32 sums over f32 activations,
    # in any order. The front end multiplies convolution inputs split in two
    # 16-bit terms. A decoder with a q8 cache rounds each new key and value to
    # 8 bits, where a last-bit difference moves a code by one, and every later
    # layer and position sees it (a prompt's whole cache is new rows); over an
    # f32 cache only the rounding of sums travels.
    if case["kind"] in ("prefill", "steps"):
        if case["cache"] == "f32":
            return {"rel": 2e-5, "max": 2e-4}
        return {"rel": 3e-2, "max": 0.2} if case["kind"] == "prefill" else {"rel": 3e-3, "max": 3e-2}
    if case["kind"] == "frontend":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 4e-6, "max": 4e-5}
