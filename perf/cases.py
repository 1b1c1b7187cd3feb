"""Performance cases of the framework: the calls that its users' programs make,
through the public entry points (pixelina_amd.Session over the C ABI, and
pixelina_amd.zimage.ZBlock for a whole transformer block).

Families (`kind`):

  linear     pixhip_matmul: y[M][N] = x[M][K] . W[N][K]^T with quantized weights.
             M = 1 is a chat decode step, M up to 128 a prompt or one chunk of a
             chat prefill, thousands of rows a diffusion transformer's tokens.
  ffn_down   pixhip_silu_gate_quantize then the multiply stage: the SwiGLU product
             and the down projection of a transformer block.
  attention  pixhip_attention_ranges: self-attention of a diffusion transformer
             (rows = keys), a decode step against the key/value cache (one row),
             a prefill chunk behind a cache (causal, offset), a VAE's single wide
             head.
  conv       pixhip_conv2d: the VAE's convolutions.
  groupnorm  pixhip_groupnorm: the VAE's norms.
  block      one Z-Image DiT block (ZBlock).

Every state has a session of its own; all sessions run on one stream, in order.
Weights are resident before the first timed pass, as they are in a program that
denoises or decodes step after step: prepare() makes one call of the case's own
shape on other data.  Outputs are device tensors over the session's buffers.
"""
import math

import numpy as np
import torch

from pixelina_amd import Q5_K, Q6_K, Q8_0, Session, _lib
from pixelina_amd.zimage import HEAD_DIM, HEADS, HIDDEN, INTERMEDIATE, NORM_EPSILON, TIME_DIM, ZBlock, ZBlockWeights, rotary

TYPES = {"q8_0": Q8_0, "q5_K": Q5_K, "q6_K": Q6_K}
BLOCK = {"q8_0": (32, 34), "q5_K": (256, 176), "q6_K": (256, 210)}
FLOAT_TYPES = {"f32": (0, 4), "f16": (1, 2), "bf16": (30, 2)}
EPSILON_GROUPNORM = 1e-6


def listed():
    return [
        # one chat decode step's widest projection
        {"name": "decode_q5_K", "kind": "linear", "type": "q5_K", "m": 1, "k": 3584, "n": 18944},
        # a short prompt through an LM's down projection, K-quant files' wider type
        {"name": "prompt_q6_K", "kind": "linear", "type": "q6_K", "m": 37, "k": 12288, "n": 4096},
        # one 128-token chunk of a chat prefill through a gate / up projection
        {"name": "prefill_q5_K", "kind": "linear", "type": "q5_K", "m": 128, "k": 4096, "n": 12288},
        # a text encoder's or refiner's linear: 256 tokens
        {"name": "linear_q8_0", "kind": "linear", "type": "q8_0", "m": 256, "k": 3840, "n": 3840},
        # the diffusion transformer's FFN up projection at 1024 x 1024 pixels
        {"name": "dit_ffn_q5_K", "kind": "linear", "type": "q5_K", "m": 4096, "k": 3840, "n": 10240},
        # its SwiGLU product and down projection, with the text tokens
        {"name": "dit_ffn_down_q8_0", "kind": "ffn_down", "type": "q8_0", "m": 4608, "k": 10240, "n": 3840},
        # its self-attention
        {"name": "dit_attention", "kind": "attention", "rows": 4608, "keys": 4608, "heads": 30, "kv_heads": 30, "dim": 128, "causal": False},
        # a chat decode step against its key/value cache (grouped heads)
        {"name": "decode_attention", "kind": "attention", "rows": 1, "keys": 2501, "heads": 32, "kv_heads": 8, "dim": 128, "causal": True},
        # a prefill chunk behind the cache of the chunks before it
        {"name": "prefill_attention", "kind": "attention", "rows": 128, "keys": 1281, "heads": 32, "kv_heads": 8, "dim": 128, "causal": True},
        # a VAE decoder's wide convolution at a quarter of the output's side
        {"name": "vae_conv", "kind": "conv", "type": "f16", "width": 256, "height": 256, "cin": 512, "cout": 512, "kernel": 3, "down": False},
        # a VAE decoder's norm at the output's size
        {"name": "vae_groupnorm", "kind": "groupnorm", "rows": 1 << 20, "channels": 128},
        # one whole block of the diffusion transformer
        {"name": "dit_block", "kind": "block", "rows": 4608, "modulated": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["ffn_down", "attention", "attention", "attention", "conv", "conv", "groupnorm", "block"])
    if kind in ("linear", "ffn_down"):
        # decode, prompts and prefill chunks, image tokens; ragged everywhere
        wtype = rng.choice(sorted(TYPES))
        m = rng.choice([1, _log(rng, 2, 128), _log(rng, 2, 4608), _log(rng, 128, 4608)]) if kind == "linear" else _log(rng, 1, 4608)
        k = 256 * _log(rng, 2, 48) if wtype != "q8_0" else 32 * _log(rng, 8, 384)
        n = _log(rng, 64, 18944)
        while 2.0 * m * n * k > 3.6e11:
            m = max(1, m // 2)
        return {"kind": kind, "type": wtype, "m": m, "k": k, "n": n}
    if kind == "attention":
        use = rng.choice(["self", "decode", "chunk", "wide"])
        if use == "wide":
            n = _log(rng, 256, 16384)
            return {"kind": kind, "rows": n, "keys": n, "heads": 1, "kv_heads": 1, "dim": rng.choice([384, 512]), "causal": False}
        kv = rng.choice([1, 2, 4, 8, 16])
        heads = kv * rng.choice([1, 2, 4, 7]) if kv <= 8 else kv
        dim = rng.choice([64, 72, 80, 128, 128])
        if use == "self":
            n = _log(rng, 32, 4608)
            return {"kind": kind, "rows": n, "keys": n, "heads": heads, "kv_heads": kv, "dim": dim, "causal": rng.random() < 0.3}
        rows = 1 if use == "decode" else rng.choice([128, _log(rng, 2, 128)])
        return {"kind": kind, "rows": rows, "keys": rows + _log(rng, 16, 16384), "heads": heads, "kv_heads": kv, "dim": dim, "causal": True}
    if kind == "conv":
        # decoder and encoder layers: the first one has few channels, the last one few outputs
        cin, cout = rng.choice([(16, 384), (16, 512), (3, 96), (3, 128), (512, 512), (384, 384), (512, 256), (192, 192), (256, 128), (128, 128),
                                (96, 96), (128, 3), (96, 3)])
        w, h = _log(rng, 24, 512), _log(rng, 24, 512)
        kernel = rng.choice([1, 3, 3, 3])
        while 2.0 * w * h * cin * cout * kernel * kernel > 3.6e11:
            w, h = w // 2 + 1, h // 2 + 1
        return {"kind": kind, "type": rng.choice(sorted(FLOAT_TYPES)), "width": w, "height": h, "cin": cin, "cout": cout, "kernel": kernel,
                "down": kernel == 3 and rng.random() < 0.25}
    if kind == "groupnorm":
        return {"kind": kind, "rows": _log(rng, 1024, 1 << 20), "channels": rng.choice([64, 96, 128])} if rng.random() < 0.5 else \
            {"kind": kind, "rows": _log(rng, 256, 1 << 18), "channels": rng.choice([256, 384, 512])}
    return {"kind": "block", "rows": 32 * _log(rng, 1, 144), "modulated": rng.random() < 0.75}


# ---- the state of a user's program ----

_streams = []


def _stream():
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


class _Owner:
    """A session that lives as long as anything that refers to its memory."""

    def __init__(self):
        self.session = Session(0)
        _lib.check(self.session.lib.pixhip_session_set_stream(self.session.handle, _stream().cuda_stream), "pixhip_session_set_stream")

    def __del__(self):
        self.session.close()


class _Memory:
    """One float32 buffer of a session, as torch sees it."""

    def __init__(self, owner, shape):
        self.owner = owner
        self.buffer = owner.session.alloc(max(4, 4 * int(np.prod(shape))))
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (self.buffer.ptr, False), "version": 2}


def _tensor(owner, shape, values=None):
    t = torch.as_tensor(_Memory(owner, shape), device="cuda")
    if values is not None:
        t.copy_(values)
    return t


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _activations(g, rows, k):
    """N(0, 1) with 1% of the channels 20 times as large, as transformers have them."""
    x = _normal(g, (rows, k))
    big = torch.randperm(k, generator=g, device="cuda")[: max(1, round(0.01 * k))]
    x[:, big] *= 20
    return x


# ---- quantized weights: GGUF blocks of about N(0, std^2) values ----


def _integers(g, lo, hi, shape):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32)


def _half_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _spread(g, shape):
    """Block scales vary by about a factor of two over a real tensor."""
    return torch.exp(_normal(g, shape, 0.25))


def _q8_0(g, n, k, std):
    b = (n, k // 32)
    d = std * 2.4 / 127 * _spread(g, b)
    q = (_normal(g, (*b, 32)) * (127 / 2.4)).round().clamp(-127, 127).to(torch.int8)
    return torch.cat([_half_bytes(d), q.view(torch.uint8)], dim=-1)


def _q5_K(g, n, k, std):
    b = (n, k // 256)
    sc = _integers(g, 24, 64, (*b, 8))
    mn = (sc + _integers(g, -4, 5, (*b, 8))).clamp(0, 63)
    d = std / 6.0 / 44 * _spread(g, b)
    q = (_normal(g, (*b, 8, 32)) * 6.0 + 15.5).round().clamp(0, 31).to(torch.int32)
    out = torch.zeros((*b, 176), dtype=torch.uint8, device="cuda")
    out[..., 0:2], out[..., 2:4] = _half_bytes(d), _half_bytes(15.5 * d)
    out[..., 4:8] = (sc[..., :4] | ((sc[..., 4:] >> 4) << 6)).to(torch.uint8)
    out[..., 8:12] = (mn[..., :4] | ((mn[..., 4:] >> 4) << 6)).to(torch.uint8)
    out[..., 12:16] = ((sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)).to(torch.uint8)
    bit = torch.arange(8, device="cuda", dtype=torch.int32)[:, None]
    out[..., 16:48] = ((q >> 4) << bit).sum(dim=-2).to(torch.uint8)
    out[..., 48:] = ((q[..., 0::2, :] & 15) | ((q[..., 1::2, :] & 15) << 4)).reshape(*b, 128).to(torch.uint8)
    return out


def _q6_K(g, n, k, std):
    b = (n, k // 256)
    sc = _integers(g, 60, 128, (*b, 16)) * (1 - 2 * _integers(g, 0, 2, (*b, 16)))
    d = std / 12.0 / 95 * _spread(g, b)
    q = (_normal(g, (*b, 2, 4, 32)) * 12.0 + 32).round().clamp(0, 63).to(torch.int32)
    out = torch.zeros((*b, 210), dtype=torch.uint8, device="cuda")
    lo = torch.stack([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], dim=-2)
    out[..., 0:128] = lo.reshape(*b, 128).to(torch.uint8)
    shift = 2 * torch.arange(4, device="cuda", dtype=torch.int32)[:, None]
    out[..., 128:192] = ((q >> 4) << shift).sum(dim=-2).reshape(*b, 64).to(torch.uint8)
    out[..., 192:208] = sc.to(torch.int8).view(torch.uint8)
    out[..., 208:210] = _half_bytes(d)
    return out


_PACK = {"q8_0": _q8_0, "q5_K": _q5_K, "q6_K": _q6_K}


def _weight_bytes(g, wtype, n, k, std=0.02):
    return _PACK[wtype](g, n, k, std).reshape(n, -1)


def _linear_inputs(case, seed):
    g = _generator(seed)
    x = _activations(g, case["m"], case["k"])
    return x, _weight_bytes(g, case["type"], case["n"], case["k"])


def _ffn_inputs(case, seed):
    g = _generator(seed)
    gate, up = _normal(g, (case["m"], case["k"]), 1.5), _normal(g, (case["m"], case["k"]))
    return gate, up, _weight_bytes(g, case["type"], case["n"], case["k"])


def _attention_inputs(case, seed):
    g = _generator(seed)
    q = _normal(g, (case["rows"], case["heads"] * case["dim"]))
    return q, _normal(g, (case["keys"], case["kv_heads"] * case["dim"])), _normal(g, (case["keys"], case["kv_heads"] * case["dim"]))


def _conv_inputs(case, seed):
    g = _generator(seed)
    c, k = case["cin"], case["kernel"]
    x = _normal(g, (case["height"] * case["width"], c))
    w = _normal(g, (case["cout"], c, k, k), 1 / math.sqrt(c * k * k))
    w = w.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[case["type"]])
    return x, w, _normal(g, (case["cout"],), 0.1)


def _conv_geometry(case):
    """(stride_x, stride_y, left, right, top, bottom): the encoder's downsampling pads on one side."""
    return (2, 2, 0, 1, 0, 1) if case["down"] else None


def _conv_out(case):
    w, h = case["width"], case["height"]
    return ((w + 1 - 3) // 2 + 1, (h + 1 - 3) // 2 + 1) if case["down"] else (w, h)


def _groupnorm_inputs(case, seed):
    g = _generator(seed)
    c = case["channels"]
    x = _normal(g, (case["rows"], c)) * (1 + torch.rand(c, generator=g, device="cuda")) + _normal(g, (c,), 0.5)
    return x, 1 + _normal(g, (c,), 0.1), _normal(g, (c,), 0.1)


_BLOCK_TYPES = {"qkv": "q5_K", "out": "q5_K", "w1": "q5_K", "w3": "q5_K", "w2": "q8_0", "modulation": "q8_0"}
_BLOCK_VECTORS = {"attention_norm1": HIDDEN, "attention_norm2": HIDDEN, "ffn_norm1": HIDDEN, "ffn_norm2": HIDDEN, "q_norm": HEAD_DIM,
                  "k_norm": HEAD_DIM}


def _block_inputs(case, seed):
    g = _generator(seed)
    keys = [k for k in _BLOCK_TYPES if k != "modulation" or case["modulated"]]
    linears = {}
    for key in keys:
        inner, rows = ZBlockWeights.SHAPES[key]
        linears[key] = _weight_bytes(g, _BLOCK_TYPES[key], rows, inner)
    vectors = {key: 1 + _normal(g, (n,), 0.1) for key, n in _BLOCK_VECTORS.items()}
    if case["modulated"]:
        vectors["modulation_bias"] = _normal(g, (4 * HIDDEN,), 0.1)
    x = _normal(g, (case["rows"], HIDDEN))
    side = max(1, math.isqrt(case["rows"]))
    cos, sin = (torch.from_numpy(t).cuda() for t in rotary(case["rows"], 32, side, case["modulated"]))
    return linears, vectors, x, cos, sin, _normal(g, (1, TIME_DIM))


def prepare(case, seed):
    owner = _Owner()
    s, kind = owner.session, case["kind"]
    state = {"case": case, "owner": owner}
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        state["x"] = _tensor(owner, x.shape, x)
        state["w"] = s.weight("w", w.cpu().numpy(), TYPES[case["type"]], case["k"], case["n"])
        state["y"] = _tensor(owner, (case["m"], case["n"]))
        other = _tensor(owner, x.shape, torch.zeros_like(x))
        torch.cuda.synchronize()
        _lib.check(s.matmul(state["w"], other.data_ptr(), case["m"], state["y"].data_ptr()), "pixhip_matmul")
    elif kind == "ffn_down":
        gate, up, w = _ffn_inputs(case, seed)
        state["gate"], state["up"] = _tensor(owner, gate.shape, gate), _tensor(owner, up.shape, up)
        state["w"] = s.weight("w", w.cpu().numpy(), TYPES[case["type"]], case["k"], case["n"])
        state["y"] = _tensor(owner, (case["m"], case["n"]))
        torch.cuda.synchronize()
        _lib.check(s.silu_gate_quantize(TYPES[case["type"]], state["up"].data_ptr(), state["up"].data_ptr(), case["m"], case["k"]), "warm")
        _lib.check(s.matmul_stage(state["w"], None, case["m"], state["y"].data_ptr(), _lib.STAGE_MULTIPLY), "warm")
    elif kind == "attention":
        for key, t in zip("qkv", _attention_inputs(case, seed)):
            state[key] = _tensor(owner, t.shape, t)
        state["out"] = _tensor(owner, state["q"].shape)
    elif kind == "conv":
        x, w, bias = _conv_inputs(case, seed)
        state["x"], state["bias"] = _tensor(owner, x.shape, x), _tensor(owner, bias.shape, bias)
        raw = w.cpu().contiguous().view(torch.uint8).reshape(-1).numpy()
        state["w"] = s.conv_weight("w", raw, FLOAT_TYPES[case["type"]][0], case["kernel"], case["kernel"], case["cin"], case["cout"])
        ow, oh = _conv_out(case)
        state["y"] = _tensor(owner, (ow * oh, case["cout"]))
        other = _tensor(owner, x.shape, torch.zeros_like(x))
        torch.cuda.synchronize()
        _lib.check(s.conv2d(state["w"], other.data_ptr(), case["width"], case["height"], state["y"].data_ptr(), _conv_geometry(case),
                            state["bias"].data_ptr()), "pixhip_conv2d")
    elif kind == "groupnorm":
        x, w, b = _groupnorm_inputs(case, seed)
        state["x"], state["w"], state["b"] = _tensor(owner, x.shape, x), _tensor(owner, w.shape, w), _tensor(owner, b.shape, b)
        state["y"] = _tensor(owner, x.shape)
    else:
        linears, vectors, x, cos, sin, time = _block_inputs(case, seed)
        weights = ZBlockWeights(s, "block", {k: (w.cpu().numpy(), TYPES[_BLOCK_TYPES[k]]) for k, w in linears.items()},
                                {k: v.cpu().numpy() for k, v in vectors.items()})
        state["weights"] = weights
        state["block"] = ZBlock(s, weights, case["rows"])
        state["x0"], state["x"] = _tensor(owner, x.shape, x), _tensor(owner, x.shape, torch.zeros_like(x))
        state["cos"], state["sin"], state["time"] = (_tensor(owner, t.shape, t) for t in (cos, sin, time))
        torch.cuda.synchronize()
        _run_block(state)
    torch.cuda.synchronize()
    return state


def _run_block(state):
    s = state["owner"].session
    # the block updates the token stream in place: each pass starts from the stream as it came in
    s.copy_device(state["x"].data_ptr(), state["x0"].data_ptr(), state["x"].numel() * 4)
    state["block"].run(state["x"].data_ptr(), state["cos"].data_ptr(), state["sin"].data_ptr(),
                       state["time"].data_ptr() if state["case"]["modulated"] else None)
    return state["x"]


def run(state):
    case = state["case"]
    s, kind = state["owner"].session, case["kind"]
    if kind == "linear":
        _lib.check(s.matmul(state["w"], state["x"].data_ptr(), case["m"], state["y"].data_ptr()), "pixhip_matmul")
        return state["y"]
    if kind == "ffn_down":
        _lib.check(s.silu_gate_quantize(TYPES[case["type"]], state["gate"].data_ptr(), state["up"].data_ptr(), case["m"], case["k"]),
                   "pixhip_silu_gate_quantize")
        _lib.check(s.matmul_stage(state["w"], None, case["m"], state["y"].data_ptr(), _lib.STAGE_MULTIPLY), "pixhip_matmul_stage")
        return state["y"]
    if kind == "attention":
        rows, keys, heads = case["rows"], case["keys"], case["heads"]
        _lib.check(s.attention(state["q"].data_ptr(), rows, state["k"].data_ptr(), state["v"].data_ptr(), keys, heads, case["kv_heads"],
                               heads * case["dim"], state["out"].data_ptr(), ranges=[(0, rows, keys, int(case["causal"]))],
                               query_offset=keys - rows), "pixhip_attention_ranges")
        return state["out"]
    if kind == "conv":
        _lib.check(s.conv2d(state["w"], state["x"].data_ptr(), case["width"], case["height"], state["y"].data_ptr(), _conv_geometry(case),
                            state["bias"].data_ptr()), "pixhip_conv2d")
        return state["y"]
    if kind == "groupnorm":
        _lib.check(s.groupnorm(state["x"].data_ptr(), case["rows"], case["channels"], state["w"].data_ptr(), state["b"].data_ptr(),
                               state["y"].data_ptr()), "pixhip_groupnorm")
        return state["y"]
    return _run_block(state)


# ---- what a pass cannot do without ----


def _gguf_bytes(wtype, n, k):
    values, nbytes = BLOCK[wtype]
    return n * (k // values) * nbytes


def _attention_pairs(rows, keys, causal):
    """Query-key pairs that are visible when query row r sees keys 0 .. keys - rows + r."""
    return rows * (keys - rows) + rows * (rows + 1) // 2 if causal else rows * keys


def work(case):
    kind = case["kind"]
    if kind in ("linear", "ffn_down"):
        m, n, k = case["m"], case["n"], case["k"]
        inputs = (1 if kind == "linear" else 2) * 4 * m * k
        return {"bytes": _gguf_bytes(case["type"], n, k) + inputs + 4 * m * n, "flops": 2.0 * m * n * k}
    if kind == "attention":
        rows, keys, h, kv, d = (case[x] for x in ("rows", "keys", "heads", "kv_heads", "dim"))
        return {"bytes": 4 * d * (2 * rows * h + 2 * keys * kv), "flops": 4.0 * h * d * _attention_pairs(rows, keys, case["causal"])}
    if kind == "conv":
        ow, oh = _conv_out(case)
        taps = case["cin"] * case["cout"] * case["kernel"] ** 2
        return {"bytes": 4 * case["width"] * case["height"] * case["cin"] + FLOAT_TYPES[case["type"]][1] * taps + 4 * ow * oh * case["cout"],
                "flops": 2.0 * ow * oh * taps}
    if kind == "groupnorm":
        return {"bytes": 8 * case["rows"] * case["channels"], "flops": 0}
    rows = case["rows"]
    total = 8 * rows * HIDDEN
    flops = 4.0 * HIDDEN * rows * rows
    for key, wtype in _BLOCK_TYPES.items():
        if key != "modulation" or case["modulated"]:
            inner, outer = ZBlockWeights.SHAPES[key]
            total += _gguf_bytes(wtype, outer, inner)
            flops += 2.0 * (1 if key == "modulation" else rows) * inner * outer
    return {"bytes": total, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "ffn_down"):
        # exact integer block sums, fp32 sums over the blocks
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "attention":
        # products of fp32 operands at about 2^-16, fp32 softmax
        return {"rel": 3e-5, "max": 1.2e-3}
    if kind == "conv":
        return {"rel": 2e-5, "max": 1e-3}
    if kind == "groupnorm":
        # double statistics; an output moves by an ulp where they meet an fp32 rounding boundary
        return {"rel": 1e-6, "max": 1e-5}
    # rounding in one op moves values over quantization steps of the next ops' inputs
    return {"rel": 1e-2}


# ---- the same in 64 bits ----


def _decode_q8_0(raw):
    b = raw.reshape(raw.shape[0], -1, 34)
    return (b[..., :2].contiguous().view(torch.float16).double() * b[..., 2:].contiguous().view(torch.int8).double()).reshape(raw.shape[0], -1)


def _decode_q5_K(raw):
    b = raw.reshape(raw.shape[0], -1, 176)
    d, dmin = (b[..., i:i + 2].contiguous().view(torch.float16).double() for i in (0, 2))
    s = b[..., 4:16].to(torch.int32)
    sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], dim=-1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], dim=-1)
    qs = b[..., 48:].to(torch.int32).reshape(*b.shape[:2], 4, 32)
    low = torch.stack([qs & 15, qs >> 4], dim=-2).reshape(*b.shape[:2], 8, 32)
    bit = torch.arange(8, device=raw.device, dtype=torch.int32)[:, None]
    q = low + (((b[..., None, 16:48].to(torch.int32) >> bit) & 1) << 4)
    return ((d * sc)[..., None] * q - (dmin * mn)[..., None]).reshape(raw.shape[0], -1)


def _decode_q6_K(raw):
    b = raw.reshape(raw.shape[0], -1, 210)
    lo = b[..., :128].to(torch.int32).reshape(*b.shape[:2], 2, 2, 32)
    low = torch.cat([lo & 15, lo >> 4], dim=-2)
    shift = 2 * torch.arange(4, device=raw.device, dtype=torch.int32)[:, None]
    high = (b[..., 128:192].to(torch.int32).reshape(*b.shape[:2], 2, 1, 32) >> shift) & 3
    q = (low + (high << 4) - 32).reshape(*b.shape[:2], 16, 16)
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    d = b[..., 208:].contiguous().view(torch.float16).double()
    return ((d * sc)[..., None] * q).reshape(raw.shape[0], -1)


_DECODE = {"q8_0": _decode_q8_0, "q5_K": _decode_q5_K, "q6_K": _decode_q6_K}


def _quantized(x, wtype):
    """The activations as the layer defines them (fp32 scales, whole-number values), widened: the
    K-quants' blocks of 256 scaled by -127 / (the first value of largest magnitude), rounded to even;
    Q8_0's blocks of 32 scaled by 127 / (the largest magnitude), rounded half away from zero, with a
    16-bit scale.  Products and quotients of fp32 values rounded once, through 64 bits."""
    if wtype == "q8_0":
        b = x.reshape(x.shape[0], -1, 32)
        d = (b.abs().amax(dim=-1, keepdim=True).double() / 127).float()
        inverse = torch.where(d > 0, (1 / d.double()).float(), torch.zeros_like(d))
        v = (b.double() * inverse.double()).float().double()
        q = torch.sign(v) * torch.floor(v.abs() + 0.5)
        return (d.half().double() * q).reshape(x.shape)
    b = x.reshape(x.shape[0], -1, 256)
    largest = b.abs().amax(dim=-1, keepdim=True)
    first = (b.abs() == largest).to(torch.uint8).argmax(dim=-1, keepdim=True)
    top = torch.gather(b, -1, first)
    scale = (-127 / top.double()).float()
    q = torch.round(scale.double() * b.double()).clamp(max=127)
    d = (1 / scale.double()).float().double()
    return torch.where(top == 0, torch.zeros_like(q), d * q).reshape(x.shape)


def _linear64(x, raw, wtype):
    return _quantized(x, wtype) @ _DECODE[wtype](raw).T


def _gated(gate, up):
    """v / (1 + e^-v) * u in fp32, each step rounded once."""
    e = torch.exp(-gate.double()).float()
    v = (gate.double() / (1.0 + e.double()).float().double()).float()
    return (v.double() * up.double()).float()


def _attention64(q, k, v, heads, kv_heads, causal):
    rows, keys = q.shape[0], k.shape[0]
    dim = q.shape[1] // heads
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 27) // keys)
    for h in range(heads):
        at = h // (heads // kv_heads) * dim
        kh, vh = k[:, at:at + dim].double(), v[:, at:at + dim].double()
        for r in range(0, rows, step):
            part = q[r:r + step, h * dim:(h + 1) * dim].double() @ kh.T / math.sqrt(dim)
            if causal:
                limit = torch.arange(r, r + part.shape[0], device=q.device)[:, None] + (keys - rows)
                part = part.masked_fill(torch.arange(keys, device=q.device)[None] > limit, -math.inf)
            out[r:r + step, h * dim:(h + 1) * dim] = torch.softmax(part, dim=-1) @ vh
    return out


def _conv64(case, x, w, bias):
    width, height, c, k = case["width"], case["height"], case["cin"], case["kernel"]
    left = 0 if case["down"] else k // 2
    stride = 2 if case["down"] else 1
    ow, oh = _conv_out(case)
    image = torch.nn.functional.pad(x.double().reshape(height, width, c), (0, 0, left, k, left, k))
    out = bias.double().expand(oh * ow, -1).clone()
    for dy in range(k):
        for dx in range(k):
            tap = image[dy:dy + stride * oh:stride, dx:dx + stride * ow:stride]
            out += tap[:oh, :ow].reshape(oh * ow, c) @ w[:, :, dy, dx].double().T
    return out


def _norm64(x, weight):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + NORM_EPSILON) * weight.double()


def _block64(case, seed):
    linears, v, x, cos, sin, time = _block_inputs(case, seed)
    rows, x = case["rows"], x.double()
    part = torch.zeros(4, HIDDEN, dtype=torch.float64, device="cuda")
    gated = case["modulated"]
    if gated:
        part = (_linear64(time, linears["modulation"], "q8_0") + v["modulation_bias"].double()).reshape(4, HIDDEN)

    def linear(key, a):
        return _linear64(a.float(), linears[key], _BLOCK_TYPES[key])

    def head(a, key):
        a = _norm64(a.reshape(rows, HEADS, HEAD_DIM), v[key]).reshape(rows, HEADS, HEAD_DIM // 2, 2)
        c, s = cos.double()[:, None], sin.double()[:, None]
        return torch.stack([a[..., 0] * c - a[..., 1] * s, a[..., 0] * s + a[..., 1] * c], dim=-1).reshape(rows, HIDDEN)

    q, k, val = linear("qkv", _norm64(x, v["attention_norm1"]) * (1 + part[0])).split(HIDDEN, dim=1)
    a = _attention64(head(q, "q_norm"), head(k, "k_norm"), val, HEADS, HEADS, False)
    x = x + _norm64(linear("out", a), v["attention_norm2"]) * (torch.tanh(part[1]) if gated else 1)
    h = _norm64(x, v["ffn_norm1"]) * (1 + part[2])
    h = _norm64(linear("w2", _gated(linear("w1", h).float(), linear("w3", h).float())), v["ffn_norm2"])
    return x + h * (torch.tanh(part[3]) if gated else 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        return _linear64(x, w, case["type"])
    if kind == "ffn_down":
        gate, up, w = _ffn_inputs(case, seed)
        return _linear64(_gated(gate, up), w, case["type"])
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        return _attention64(q, k, v, case["heads"], case["kv_heads"], case["causal"])
    if kind == "conv":
        return _conv64(case, *_conv_inputs(case, seed))
    if kind == "groupnorm":
        x, w, b = _groupnorm_inputs(case, seed)
        rows, c = x.shape
        g = x.double().reshape(rows, 32, c // 32)
        mean = g.mean(dim=(0, 2), keepdim=True)
        variance = (g - mean).square().mean(dim=(0, 2), keepdim=True)
        return ((g - mean) * torch.rsqrt(variance + EPSILON_GROUPNORM)).reshape(rows, c) * w.double() + b.double()
    return _block64(case, seed)


assert INTERMEDIATE == ZBlockWeights.SHAPES["w2"][0]
