"""Timed cases of the framework's public entry points: the work a RoFormer separation program
gives them, from single ops on the smallest calls up to whole clips.

Every case is a dict of plain values with an ``op``:

  attention  fused.attention            softmax(q k^T) v per (group, head), optional rotary table
  gated      fused.gated_attention      the same from one packed q | k | v | gates projection
  linear     fused.linear / norm_linear a block's projections with their epilogues
  unit_norm  fused.unit_norm            the row norm (with the final norm's scale)
  block      roformer.Transformer       one transformer block
  pair       roformer.AxisPair          time pass + band pass of the axis loop
  stft/istft separation.stft / istft    both channels of a clip, and back through a mask
  separate   separation.Roformer        a whole clip through a model

``listed`` gives the fixed cases, ``draw`` one more of the same ranges, ``prepare`` / ``run`` the
inputs and one pass, ``exact`` the outputs in float64 from plain torch, ``work`` the bytes and
operations of a pass and ``tolerance`` the agreement two correct implementations reach.
"""
import math

import torch

from ancha_amd import fused, roformer, separation

DEVICE = "cuda"
HEAD = 64
N_FFT = 2048
BINS = N_FFT // 2 + 1
HOP = 441
RATE = 44100
# Widest rows x tokens of one op call in the bundled models: two chunks of 60 bands x 801 frames.
MAX_ROWS = 110_000


def listed():
    return [
        # The time pass of two 8 s chunks of the bundled Mel model, rotary table on load.
        {"name": "attention_time", "op": "attention", "groups": 120, "tokens": 801, "heads": 8,
         "rope": True},
        # A chunk of the longest sequences the op is quoted on: 90 bands x 1722 frames, q and k
        # already rotated.
        {"name": "attention_1722", "op": "attention", "groups": 90, "tokens": 1722, "heads": 8,
         "rope": False},
        # A small call (four sequences of 256 tokens): launch and latency, a nearly idle chip.
        {"name": "attention_small", "op": "attention", "groups": 4, "tokens": 256, "heads": 2,
         "rope": False},
        # The band pass of two 8 s chunks on the packed projection (60 bands per frame).
        {"name": "gated_band", "op": "gated", "groups": 1602, "tokens": 60, "heads": 8,
         "columns": 1664, "rope": False},
        # The block's first projection over two chunks: row norm, bias, rotary epilogue.
        {"name": "linear_qkv", "op": "linear", "kind": "qkv", "groups": 120, "tokens": 801,
         "dim": 384, "heads": 8},
        # The feed-forward's second projection over one 3 s chunk (60 bands x 301 frames): the
        # long k, bias and residual.
        {"name": "linear_ff_out", "op": "linear", "kind": "ff_out", "groups": 60, "tokens": 301,
         "dim": 384, "heads": 8},
        # The norm between layers over two chunks.
        {"name": "unit_norm", "op": "unit_norm", "rows": 96120, "dim": 384, "scaled": True},
        # One time block over a 3 s chunk.
        {"name": "block_3s", "op": "block", "groups": 60, "tokens": 301, "dim": 384, "heads": 8,
         "output_norm": True},
        # One layer pair over two 8 s chunks: the bulk of a separation.
        {"name": "layer_pair", "op": "pair", "batch": 2, "bands": 60, "frames": 801, "dim": 384,
         "heads": 8, "output_norm": True},
        # Analysis of a 30 s clip.
        {"name": "stft_30s", "op": "stft", "samples": 30 * RATE, "hop": HOP},
        # Masked synthesis of one 8 s chunk (801 frames).
        {"name": "istft_8s", "op": "istft", "frames": 801, "hop": HOP, "zero_dc": True},
        # A whole clip of twelve seconds and a ragged end (thirteen 8 s chunks at overlap 4, an odd
        # count) through the bundled Mel model.
        {"name": "separate_12s", "op": "separate", "family": "mel", "dim": 384, "depth": 6,
         "heads": 8, "samples": 533_001},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    op = rng.choice(["attention", "attention", "gated", "linear", "linear", "unit_norm", "block",
                     "block", "pair", "stft", "istft", "separate"])
    if op == "attention":
        tokens = _log(rng, 16, 1722)
        return {"op": op, "tokens": tokens, "groups": _log(rng, 1, min(1602, MAX_ROWS // tokens)),
                "heads": rng.choice([1, 2, 3, 4, 8, 8, 8]), "rope": rng.random() < 0.5}
    if op == "gated":
        tokens, heads = _log(rng, 16, 1301), rng.choice([1, 2, 4, 8, 8, 8])
        # The packed width: padded to 128 columns, or bare with a few odd columns behind.
        bare = heads * (3 * HEAD + 1)
        columns = -(-bare // 128) * 128 if rng.random() < 0.75 else bare + rng.randrange(6)
        return {"op": op, "tokens": tokens, "groups": _log(rng, 1, min(1602, MAX_ROWS // tokens)),
                "heads": heads, "columns": columns, "rope": rng.random() < 0.5}
    if op == "linear":
        dim, tokens = rng.choice([128, 256, 384, 512]), _log(rng, 16, 1301)
        return {"op": op, "kind": rng.choice(["qkv", "out", "ff_in", "ff_out"]),
                "groups": _log(rng, 1, MAX_ROWS // tokens), "tokens": tokens, "dim": dim,
                "heads": 2 if dim == 128 else 8}
    if op == "unit_norm":
        return {"op": op, "rows": _log(rng, 1, MAX_ROWS), "scaled": rng.random() < 0.5,
                "dim": rng.choice([128, 256, 384, 512, rng.randrange(65, 1024)])}
    if op == "block":
        dim, tokens = rng.choice([128, 256, 384, 384, 512]), _log(rng, 33, 1301)
        return {"op": op, "tokens": tokens, "groups": _log(rng, 1, MAX_ROWS // tokens),
                "dim": dim, "heads": 2 if dim == 128 else 8, "output_norm": rng.random() < 0.7}
    if op == "pair":
        dim, frames = rng.choice([256, 384, 512]), _log(rng, 65, 1301)
        batch = 2 if frames <= 850 and rng.random() < 0.5 else 1
        return {"op": op, "batch": batch, "bands": rng.choice([60, 62, rng.randrange(8, 65)]),
                "frames": frames, "dim": dim, "heads": 8, "output_norm": rng.random() < 0.6}
    if op == "stft":
        return {"op": op, "samples": _log(rng, 4_000, 300 * RATE),
                "hop": rng.choice([HOP, HOP, 512, rng.randrange(256, 1025)])}
    if op == "istft":
        return {"op": op, "frames": _log(rng, 8, 3001), "zero_dc": rng.random() < 0.5,
                "hop": rng.choice([HOP, HOP, 512, rng.randrange(256, 1025)])}
    return {"op": "separate", "family": rng.choice(["mel", "bs"]), "heads": 8,
            "dim": rng.choice([256, 384]), "depth": rng.choice([1, 2]),
            "samples": _log(rng, RATE, 13 * RATE)}


# ---- inputs -----------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEVICE) * scale


def _freqs():
    return 10000.0 ** (-torch.arange(HEAD // 2, dtype=torch.float64) / (HEAD // 2))


def _rope_table(tokens):
    """The packed [4, tokens, 64] float32 table: query cos and signed sin times 1/8, key cos and
    signed sin; interleaved channel pairs."""
    freqs = _freqs().float()
    angle = (torch.arange(tokens, dtype=torch.float32)[:, None] * freqs).double()
    cos = angle.cos().repeat_interleave(2, 1)
    sin = torch.stack([-angle.sin(), angle.sin()], 2).reshape(tokens, HEAD)
    return torch.stack([cos / 8, sin / 8, cos, sin]).float().to(DEVICE)


def _audio(g, samples):
    """Stereo music-like audio [2, samples]: pink noise at 0.1 RMS plus three shared tones."""
    # A pink filter over blocks keeps the transform length a power of two whatever `samples` is.
    n = 1 << max(12, (samples - 1).bit_length())
    spec = torch.fft.rfft(_normal(g, 2, n).double())
    spec /= torch.arange(1, n // 2 + 2, device=DEVICE, dtype=torch.float64).sqrt()
    pink = torch.fft.irfft(spec, n)[:, :samples]
    pink *= 0.1 / pink.std(dim=1, keepdim=True)
    t = torch.arange(samples, device=DEVICE, dtype=torch.float64) / RATE
    pitch = _normal(g, 3).abs().double().cpu().tolist()
    for i, p in enumerate(pitch):
        pink += 0.05 * torch.sin(2 * math.pi * 110.0 * 2 ** (2 * p) * t + i)
    return pink.float().contiguous()


def _packed_columns(heads):
    return -(-heads * (3 * HEAD + 1) // 128) * 128


def _linear_shape(case):
    dim, inner = case["dim"], case["heads"] * HEAD
    return {"qkv": (dim, _packed_columns(case["heads"])), "out": (inner, dim),
            "ff_in": (dim, 4 * dim), "ff_out": (4 * dim, dim)}[case["kind"]]


def _block_weights(g, dim, heads, output_norm):
    """One block's weights in nn.Linear layout, on the GPU."""
    inner, hidden = heads * HEAD, 4 * dim
    gamma = lambda: 1.0 + _normal(g, dim, scale=0.1)
    w = {"attn_gamma": gamma(), "to_qkv": _normal(g, 3 * inner, dim, scale=0.02),
         "to_gates": _normal(g, heads, dim, scale=0.02),
         "to_gates_bias": _normal(g, heads, scale=0.02),
         "to_out": _normal(g, dim, inner, scale=0.02), "ff_gamma": gamma(),
         "ff_in": _normal(g, hidden, dim, scale=0.02), "ff_in_bias": _normal(g, hidden, scale=0.02),
         "ff_out": _normal(g, dim, hidden, scale=0.02), "ff_out_bias": _normal(g, dim, scale=0.02)}
    if output_norm:
        w["output_gamma"] = gamma()
    return w


def _config(case):
    """The bundled band layouts and DSP settings at the case's width and depth."""
    name = "mel_karaoke" if case["family"] == "mel" else "bs_roformer_large"
    return dict(separation.load_config(name), dim=case["dim"], depth=case["depth"],
                heads=case["heads"])


def _model_tensors(g, config):
    """Checkpoint tensors by name, on the GPU."""
    dim, mh = config["dim"], config["dim"] * config["mask_expansion"]
    mel = config["family"] == "mel-band-roformer"
    t = {}

    def linear(name, out, k, bias=True):
        t[name + ".weight"] = _normal(g, out, k, scale=0.02)
        if bias:
            t[name + ".bias"] = _normal(g, out, scale=0.02)

    for b, bins in enumerate(config["bands"]):
        p, width = f"band_split.to_features.{b}", 4 * len(bins)
        t[f"{p}.0.gamma"] = 1.0 + _normal(g, width, scale=0.1)
        linear(f"{p}.1", dim, width)
    for i in range(config["depth"]):
        for axis in range(2):
            p = f"layers.{i}.{axis}"
            a, f = f"{p}.layers.0.0", f"{p}.layers.0.1.net"
            w = _block_weights(g, dim, config["heads"], mel)
            for key, name in (("attn_gamma", f"{a}.norm.gamma"), ("to_qkv", f"{a}.to_qkv.weight"),
                              ("to_gates", f"{a}.to_gates.weight"),
                              ("to_gates_bias", f"{a}.to_gates.bias"),
                              ("to_out", f"{a}.to_out.0.weight"), ("ff_gamma", f"{f}.0.gamma"),
                              ("ff_in", f"{f}.1.weight"), ("ff_in_bias", f"{f}.1.bias"),
                              ("ff_out", f"{f}.4.weight"), ("ff_out_bias", f"{f}.4.bias"),
                              ("output_gamma", f"{p}.norm.gamma")):
                if key in w:
                    t[name] = w[key]
            t[f"{a}.rotary_embed.freqs"] = _freqs().float().to(DEVICE)
    if not mel:
        t["final_norm.gamma"] = 1.0 + _normal(g, dim, scale=0.1)
    hidden = config["mask_depth"] if mel else config["mask_depth"] - 1
    for s in range(len(config["stems"])):
        for b, bins in enumerate(config["bands"]):
            p = f"mask_estimators.{s}.to_freqs.{b}.0"
            for layer in range(hidden):
                linear(f"{p}.{2 * layer}", mh, dim if layer == 0 else mh)
            linear(f"{p}.{2 * hidden}", 8 * len(bins), mh)
    return t


def _inputs(case, seed):
    """The tensors of a pass, from the seed alone."""
    g, op = _generator(seed), case["op"]
    if op == "attention":
        shape = (case["groups"], case["tokens"], case["heads"], HEAD)
        # Without the table q comes scaled by 1/8, as the op takes it.
        q = _normal(g, *shape, scale=1.0 if case["rope"] else 0.125)
        return {"q": q, "k": _normal(g, *shape), "v": _normal(g, *shape),
                "rope": _rope_table(case["tokens"]) if case["rope"] else None}
    if op == "gated":
        inner = case["heads"] * HEAD
        packed = _normal(g, case["groups"], case["tokens"], case["columns"])
        if not case["rope"]:
            packed[..., :inner] *= 0.125
        packed[..., 3 * inner + case["heads"]:] = 0.0
        return {"packed": packed, "rope": _rope_table(case["tokens"]) if case["rope"] else None}
    if op == "linear":
        k, m = _linear_shape(case)
        n, kind = case["groups"] * case["tokens"], case["kind"]
        d = {"x": _normal(g, n, k, scale=0.5 if kind in ("out", "ff_out") else 2.0),
             # Weights behind a row norm carry its sqrt(dim).
             "w": _normal(g, k, m, scale=0.02 * (math.sqrt(k) if kind in ("qkv", "ff_in") else 1)),
             "bias": None if kind == "out" else _normal(g, m, scale=0.02),
             "residual": _normal(g, n, m) if kind in ("out", "ff_out") else None,
             "rope": _rope_table(case["tokens"]) if kind == "qkv" else None}
        return d
    if op == "unit_norm":
        return {"x": _normal(g, case["rows"], case["dim"], scale=2.0),
                "scale": (math.sqrt(case["dim"]) * (1.0 + _normal(g, case["dim"], scale=0.1))
                          if case["scaled"] else None)}
    if op == "block":
        return {"w": _block_weights(g, case["dim"], case["heads"], case["output_norm"]),
                "x": _normal(g, case["groups"], case["tokens"], case["dim"]),
                "rope": _rope_table(case["tokens"])}
    if op == "pair":
        w = [_block_weights(g, case["dim"], case["heads"], case["output_norm"]) for _ in range(2)]
        return {"w": w, "x": _normal(g, case["batch"], case["bands"], case["frames"], case["dim"]),
                "rope": [_rope_table(case["frames"]), _rope_table(case["bands"])]}
    if op == "stft":
        return {"audio": _audio(g, case["samples"])}
    if op == "istft":
        samples = (case["frames"] - 1) * case["hop"]
        signal = _audio(g, max(samples, N_FFT))
        spectrum = _exact_stft(signal, case["hop"])[:case["frames"]].float().contiguous()
        masks = _normal(g, 2 * BINS, 2, case["frames"], scale=0.3)
        masks[:, 0] += 0.5
        return {"spectrum": spectrum, "masks": masks, "length": samples}
    config = _config(case)
    return {"config": config, "tensors": _model_tensors(g, config),
            "audio": _audio(g, case["samples"])}


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case)
    host = lambda w, heads: {**{k: v.cpu().numpy() for k, v in w.items()}, "heads": heads}
    if case["op"] == "linear":
        table = state["rope"]
        state["epilogue"] = fused.Epilogue(
            bias=state["bias"], gelu=case["kind"] == "ff_in", residual=state["residual"],
            rotary=None if table is None else (table, case["heads"] * HEAD))
    elif case["op"] == "block":
        state["block"] = roformer.Transformer(host(state.pop("w"), case["heads"]))
    elif case["op"] == "pair":
        state["pair"] = roformer.AxisPair(*(roformer.Transformer(host(w, case["heads"]))
                                            for w in state.pop("w")))
    elif case["op"] == "separate":
        tensors = {k: v.cpu().numpy() for k, v in state.pop("tensors").items()}
        state["model"] = separation.Roformer(state["config"], tensors)
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "attention":
        return fused.attention(state["q"], state["k"], state["v"], rope=state["rope"])
    if op == "gated":
        return fused.gated_attention(state["packed"], case["heads"], rope=state["rope"])
    if op == "linear":
        call = fused.norm_linear if case["kind"] in ("qkv", "ff_in") else fused.linear
        return call(state["x"], state["w"], state["epilogue"])
    if op == "unit_norm":
        return fused.unit_norm(state["x"], state["scale"])
    if op == "block":
        return state["block"](state["x"], state["rope"])
    if op == "pair":
        return state["pair"](state["x"], *state["rope"])
    if op == "stft":
        return separation.stft(state["audio"], case["hop"])
    if op == "istft":
        return separation.istft(state["spectrum"], state["masks"], case["hop"], state["length"],
                                case["zero_dc"])
    stems, residual = state["model"].separate(state["audio"])
    return [stems] if residual is None else [stems, residual]


# ---- the work of a pass -----------------------------------------------------------------------

def _block_flops(groups, tokens, dim, heads):
    inner, hidden = heads * HEAD, 4 * dim
    per_row = 2 * dim * (3 * inner + heads) + 2 * inner * dim + 4 * dim * hidden
    return groups * tokens * (per_row + 4 * tokens * inner)


def _block_weight_bytes(dim, heads):
    inner, hidden = heads * HEAD, 4 * dim
    return 2 * (dim * (3 * inner + heads) + inner * dim + 2 * dim * hidden)  # held as fp16


def _chunk_starts(config, samples):
    step = config["chunk_samples"] // config["overlap"]
    border = config["chunk_samples"] - step
    if not samples > 2 * border:
        border = 0
    return list(range(0, samples + 2 * border, step)), border


def work(case):
    op = case["op"]
    fft = 5 * N_FFT * 11  # a complex transform of 2048 points
    if op in ("attention", "gated"):
        rows, inner = case["groups"] * case["tokens"], case["heads"] * HEAD
        bytes_ = 4 * rows * 4 * inner + (4 * case["tokens"] * HEAD * 4 if case["rope"] else 0)
        if op == "gated":
            bytes_ += 4 * rows * case["heads"]
        return {"bytes": bytes_, "flops": 4 * rows * case["tokens"] * inner}
    if op == "linear":
        k, m = _linear_shape(case)
        n = case["groups"] * case["tokens"]
        extra = n * m if case["kind"] in ("out", "ff_out") else 0
        return {"bytes": 4 * (n * k + k * m + n * m + extra), "flops": 2 * n * k * m}
    if op == "unit_norm":
        n = case["rows"] * case["dim"]
        return {"bytes": 8 * n, "flops": 3 * n}
    if op == "block":
        rows = case["groups"] * case["tokens"]
        return {"bytes": 8 * rows * case["dim"] + _block_weight_bytes(case["dim"], case["heads"]),
                "flops": _block_flops(case["groups"], case["tokens"], case["dim"], case["heads"])}
    if op == "pair":
        b, n, t, dim, heads = (case[k] for k in ("batch", "bands", "frames", "dim", "heads"))
        return {"bytes": 8 * b * n * t * dim + 2 * _block_weight_bytes(dim, heads),
                "flops": _block_flops(b * n, t, dim, heads) + _block_flops(b * t, n, dim, heads)}
    if op == "stft":
        frames = case["samples"] // case["hop"] + 1
        return {"bytes": 8 * case["samples"] + 16 * frames * BINS, "flops": frames * fft}
    if op == "istft":
        frames = case["frames"]
        return {"bytes": 32 * frames * BINS + 8 * (frames - 1) * case["hop"],
                "flops": frames * (fft + 12 * BINS)}
    config = _config(case)
    dim, heads, depth = case["dim"], case["heads"], case["depth"]
    mh, widths = dim * config["mask_expansion"], [4 * len(b) for b in config["bands"]]
    bands, frames = len(widths), config["chunk_samples"] // config["hop"] + 1
    layers = config["mask_depth"] - (config["family"] != "mel-band-roformer")
    head = [2 * (dim * mh + (layers - 1) * mh * mh + mh * 2 * w) for w in widths]
    chunk = (sum(2 * frames * dim * w for w in widths) + frames * sum(head) * len(config["stems"])
             + depth * (_block_flops(bands, frames, dim, heads)
                        + _block_flops(frames, bands, dim, heads)) + 2 * frames * fft)
    weights = (4 * dim * sum(widths) + 2 * depth * _block_weight_bytes(dim, heads)
               + sum(head) * len(config["stems"]))
    return {"bytes": weights + 4 * 2 * case["samples"] * 3,
            "flops": len(_chunk_starts(config, case["samples"])[0]) * chunk}


# ---- tolerances -------------------------------------------------------------------------------

def tolerance(case):
    """About four times the largest difference from `exact` seen over listed and drawn cases: the
    ops round their matrix operands to fp16 (2^-11 each) and accumulate in fp32; the norm and the
    transforms are fp32 throughout."""
    op = case["op"]
    if op in ("attention", "gated"):
        return {"rel": 1.7e-3, "max": 2.4e-2}
    if op == "linear":
        return {"rel": 1.2e-3, "max": 9e-3}
    if op == "unit_norm":
        return {"rel": 3e-7, "max": 1.2e-6}
    if op in ("block", "pair"):
        return {"rel": 5e-4, "max": 3e-3}
    if op == "stft":
        return {"rel": 6e-7, "max": 2.5e-5}
    if op == "istft":
        return {"rel": 5e-7, "max": 3e-6}
    return {"rel": 2.8e-3, "max": 1.3e-2}


# ---- the same results in float64 --------------------------------------------------------------

def _rotate(x, cos, sin):
    """x [..., T, H, 64] by per-token cos / signed sin rows (interleaved channel pairs)."""
    swapped = x.unflatten(-1, (-1, 2)).flip(-1).flatten(-2)
    return x * cos[:, None, :] + swapped * sin[:, None, :]


def _attend(q, k, v):
    """softmax(q k^T) v over [G, T, H, 64] float64, a few groups at a time."""
    groups, tokens, heads, _ = q.shape
    step = max(1, int(2e8 // (heads * tokens * tokens)))
    out = torch.empty_like(q)
    for a in range(0, groups, step):
        s = slice(a, min(groups, a + step))
        kt = k[s].permute(0, 2, 3, 1).contiguous()
        p = torch.softmax(torch.matmul(q[s].transpose(1, 2).contiguous(), kt), dim=-1)
        out[s] = torch.matmul(p, v[s].transpose(1, 2).contiguous()).transpose(1, 2)
    return out


def _norm(x):
    return x / torch.linalg.vector_norm(x, dim=-1, keepdim=True).clamp_min(1e-12)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _exact_block(w, heads, x):
    """One block over x [groups, tokens, dim] float64; w float64."""
    groups, tokens, dim = x.shape
    inner, root = heads * HEAD, math.sqrt(dim)
    xn = _norm(x) * root * w["attn_gamma"]
    q, k, v = ((xn @ part.t().contiguous()).view(groups, tokens, heads, HEAD)
               for part in w["to_qkv"].split(inner))
    angle = torch.arange(tokens, dtype=torch.float64)[:, None] * _freqs()
    cos = angle.cos().repeat_interleave(2, 1).to(x.device)
    sin = torch.stack([-angle.sin(), angle.sin()], 2).reshape(tokens, HEAD).to(x.device)
    o = _attend(_rotate(q, cos, sin) / 8, _rotate(k, cos, sin), v)
    gates = torch.sigmoid(xn @ w["to_gates"].t().contiguous() + w["to_gates_bias"])
    x = x + (o * gates[..., None]).view(groups, tokens, inner) @ w["to_out"].t().contiguous()
    h = _norm(x) * root * w["ff_gamma"] @ w["ff_in"].t().contiguous() + w["ff_in_bias"]
    x = x + _gelu(h) @ w["ff_out"].t().contiguous() + w["ff_out_bias"]
    return _norm(x) * root * w["output_gamma"] if "output_gamma" in w else x


def _exact_pair(weights, heads, x):
    """Time block then band block over x [batch, bands, frames, dim] float64."""
    batch, bands, frames, dim = x.shape
    x = _exact_block(weights[0], heads, x.reshape(batch * bands, frames, dim))
    x = x.view(batch, bands, frames, dim).transpose(1, 2).reshape(batch * frames, bands, dim)
    x = _exact_block(weights[1], heads, x)
    return x.view(batch, frames, bands, dim).transpose(1, 2).contiguous()


def _reflect(i, n):
    period = 2 * (n - 1)
    i = i % period
    return torch.where(i < n, i, period - i)


def _window():
    i = torch.arange(N_FFT, device=DEVICE, dtype=torch.float64)
    return 0.5 - 0.5 * torch.cos(2 * math.pi * i / N_FFT)


def _exact_stft(signal, hop):
    """[2, samples] -> [frames, 1025, 2, 2] float64 (frame, bin, channel, re/im)."""
    n = signal.shape[1]
    frames = n // hop + 1
    out = torch.empty(frames, BINS, 2, 2, dtype=torch.float64, device=DEVICE)
    x, win = signal.double(), _window()
    for a in range(0, frames, 4096):
        b = min(frames, a + 4096)
        at = torch.arange(a * hop - N_FFT // 2, (b - 1) * hop + N_FFT // 2, device=DEVICE)
        z = torch.fft.rfft(x[:, _reflect(at, n)].unfold(1, N_FFT, hop) * win)
        out[a:b] = torch.view_as_real(z).permute(1, 2, 0, 3)
    return out


def _exact_istft(spectrum, masks, hop, length, zero_dc):
    """spectrum [frames, 1025, 2, 2], masks [2050, 2, frames], float64 -> [2, length]."""
    frames = spectrum.shape[0]
    s = torch.view_as_complex(spectrum).permute(2, 0, 1)                 # [2, frames, bins]
    m = masks.view(BINS, 2, 2, frames).permute(1, 3, 0, 2).contiguous()  # [2, frames, bins, re/im]
    z = s * torch.view_as_complex(m)
    z[..., 0] = 0.0 if zero_dc else z[..., 0].real.to(z.dtype)
    z[..., -1] = z[..., -1].real.to(z.dtype)
    win = _window()
    y = torch.fft.irfft(z, N_FFT) * win
    total = (frames - 1) * hop + N_FFT
    at = torch.arange(frames, device=DEVICE)[:, None] * hop + torch.arange(N_FFT, device=DEVICE)
    acc = torch.zeros(3, total, dtype=torch.float64, device=DEVICE)
    acc[:2].index_add_(1, at.flatten(), y.reshape(2, -1))
    acc[2].index_add_(0, at.flatten(), (win * win).repeat(frames))
    return (acc[:2] / acc[2].clamp_min(1e-11))[:, N_FFT // 2:N_FFT // 2 + length]


def _exact_masks(config, t, spectrum):
    """spectrum [frames, 1025, 2, 2] float64 -> masks [stems, 2050, 2, frames]."""
    frames, mel = spectrum.shape[0], config["family"] == "mel-band-roformer"
    bands = [torch.tensor(b, device=DEVICE) for b in config["bands"]]
    f64 = lambda name: t[name].double()
    feats = []
    for b, bins in enumerate(bands):
        p = f"band_split.to_features.{b}"
        z = spectrum[:, bins].reshape(frames, -1)
        z = _norm(z) * math.sqrt(z.shape[1]) * f64(f"{p}.0.gamma")
        feats.append(z @ f64(f"{p}.1.weight").t().contiguous() + f64(f"{p}.1.bias"))
    x = torch.stack(feats)[None]
    for i in range(config["depth"]):
        blocks = []
        for axis in range(2):
            p = f"layers.{i}.{axis}"
            a, f = f"{p}.layers.0.0", f"{p}.layers.0.1.net"
            w = {"attn_gamma": f"{a}.norm.gamma", "to_qkv": f"{a}.to_qkv.weight",
                 "to_gates": f"{a}.to_gates.weight", "to_gates_bias": f"{a}.to_gates.bias",
                 "to_out": f"{a}.to_out.0.weight", "ff_gamma": f"{f}.0.gamma",
                 "ff_in": f"{f}.1.weight", "ff_in_bias": f"{f}.1.bias",
                 "ff_out": f"{f}.4.weight", "ff_out_bias": f"{f}.4.bias"}
            if mel:
                w["output_gamma"] = f"{p}.norm.gamma"
            blocks.append({k: f64(v) for k, v in w.items()})
        x = _exact_pair(blocks, config["heads"], x)
    x = x[0]
    if not mel:
        x = _norm(x) * math.sqrt(config["dim"]) * f64("final_norm.gamma")
    linears = config["mask_depth"] + (1 if mel else 0)
    masks = []
    for s in range(len(config["stems"])):
        acc = torch.zeros(BINS, 4, frames, dtype=torch.float64, device=DEVICE)
        cover = torch.zeros(BINS, dtype=torch.float64, device=DEVICE)
        for b, bins in enumerate(bands):
            h, p = x[b], f"mask_estimators.{s}.to_freqs.{b}.0"
            for layer in range(linears):
                h = h @ f64(f"{p}.{2 * layer}.weight").t().contiguous() + f64(f"{p}.{2 * layer}.bias")
                if layer + 1 < linears:
                    h = torch.tanh(h)
            value, gate = h.chunk(2, dim=1)
            acc[bins] += (value * torch.sigmoid(gate)).t().reshape(len(bins), 4, frames)
            cover[bins] += 1.0
        masks.append((acc / cover[:, None, None]).view(2 * BINS, 2, frames))
    return torch.stack(masks)


def _exact_separate(config, tensors, audio):
    n, size = audio.shape[1], config["chunk_samples"]
    starts, border = _chunk_starts(config, n)
    length, stems = n + 2 * border, len(config["stems"])
    x = audio.double()
    sums = torch.zeros(stems, 2, length, dtype=torch.float64, device=DEVICE)
    weights = torch.zeros(length, dtype=torch.float64, device=DEVICE)
    i = torch.arange(size, device=DEVICE)
    fade = max(size // 10, 1)
    for start in starts:
        remaining = min(length - start, size)
        local = torch.where(i < remaining, i, _reflect(i, remaining)) if remaining > 1 else 0 * i
        chunk = x[:, _reflect(start + local - border, n)]
        if remaining <= size // 2:
            chunk[:, remaining:] = 0.0
        spectrum = _exact_stft(chunk, config["hop"])
        masks = _exact_masks(config, tensors, spectrum)
        wt = torch.ones(size, dtype=torch.float64, device=DEVICE)
        if start > 0:
            wt[:fade] = (i[:fade] + 1) / fade
        if start + size < length:
            wt[size - fade:] = (size - i[size - fade:]) / fade
        end = min(start + size, length)
        for s in range(stems):
            y = _exact_istft(spectrum, masks[s], config["hop"], size, config["zero_dc"])
            sums[s, :, start:end] += (wt * y)[:, :end - start]
        weights[start:end] += wt[:end - start]
    out = (sums / weights)[..., border:border + n].contiguous()
    return [out, x - out[0]] if stems == 1 else [out]


def exact(case, seed):
    d, op = _inputs(case, seed), case["op"]
    if op in ("attention", "gated"):
        if op == "gated":
            inner, heads = case["heads"] * HEAD, case["heads"]
            packed = d["packed"].double()
            shape = (case["groups"], case["tokens"], heads, HEAD)
            q, k, v = (packed[..., i * inner:(i + 1) * inner].reshape(shape) for i in range(3))
        else:
            q, k, v = (d[n].double() for n in "qkv")
        if d["rope"] is not None:
            table = d["rope"].double()
            q, k = _rotate(q, table[0], table[1]), _rotate(k, table[2], table[3])
        out = _attend(q, k, v)
        if op == "gated":
            out = out * torch.sigmoid(packed[..., 3 * inner:3 * inner + heads])[..., None]
        return out
    if op == "linear":
        x, w = d["x"].double(), d["w"].double()
        y = (_norm(x) if case["kind"] in ("qkv", "ff_in") else x) @ w
        if d["bias"] is not None:
            y = y + d["bias"].double()
        if case["kind"] == "ff_in":
            y = _gelu(y)
        if d["rope"] is not None:
            table, heads = d["rope"].double(), case["heads"]
            v = y[:, :2 * heads * HEAD].reshape(case["groups"], case["tokens"], 2 * heads, HEAD)
            v = torch.cat([_rotate(v[:, :, :heads], table[0], table[1]),
                           _rotate(v[:, :, heads:], table[2], table[3])], 2)
            y[:, :2 * heads * HEAD] = v.reshape(y.shape[0], -1)
        if d["residual"] is not None:
            y = y + d["residual"].double()
        return y
    if op == "unit_norm":
        y = _norm(d["x"].double())
        return y if d["scale"] is None else y * d["scale"].double()
    double = lambda w: {k: v.double() for k, v in w.items()}
    if op == "block":
        return _exact_block(double(d["w"]), case["heads"], d["x"].double())
    if op == "pair":
        return _exact_pair([double(w) for w in d["w"]], case["heads"], d["x"].double())
    if op == "stft":
        return _exact_stft(d["audio"], case["hop"])
    if op == "istft":
        return _exact_istft(d["spectrum"].double(), d["masks"].double(), case["hop"], d["length"],
                            case["zero_dc"])
    return _exact_separate(d["config"], d["tensors"], d["audio"])
