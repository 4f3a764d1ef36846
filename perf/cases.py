"""The work that a program has this backend do, as cases that can be timed and checked.

Every case runs through the public entry points: command packets built once and submitted with
`vnpu_stream_submit`, and the decoder block of `libvnpu_block.so`.  All states share one device and stream
(a second device for the high-throughput option), as one program does, and keep their tensors in buffers of
`vnpu_buffer_alloc` that torch sees as its own.

Kinds of cases:
  linear_i8   QUANTIZE_I8 of the activations by row, then MATMUL_I8 on packed weights: a projection at decode
              (few rows), at batched decode and prompt chunks (tens to hundreds) and at prefill (thousands).
  linear_f32  MATMUL_F32 with bias and activation, weights [K][N] or [N][K], with or without an accumulated C.
  head        MTP_HEAD_F32 and SOFTMAX_F32: the logits and probabilities of a few drafted tokens.
  attention   ATTENTION_F32: prefill, a chunk of a prompt behind a cache, or decode, on either kind of device.
  block       one whole decoder layer: RMSNorm, projections, RoPE, attention, SwiGLU, residuals.
"""
import ctypes as C
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "npuxl-improved_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "npuxl-improved_amd"))

from vnpu_mi355x import Session, abi  # noqa: E402
from vnpu_mi355x import block as blk  # noqa: E402

EPILOGUES = {"none": abi.EPI_NONE, "silu": abi.EPI_SILU, "gelu": abi.EPI_GELU_TANH}
PROJECTIONS = ("qkv", "o", "gate", "up", "down")


def listed():
    return [
        # One token through a small layer (width 512, FFN 1376, 8 heads): every kernel is a few microseconds, so
        # this is launches, gaps and latency; 1376 is no multiple of 64.
        {"name": "block_decode_small", "kind": "block", "batch": 1, "tokens": 1, "past": 127, "width": 512,
         "heads": 8, "ffn": 1376},
        # One token through the largest projection of a 4096-wide model, its output head: the weight stream.
        {"name": "i8_decode_head", "kind": "linear_i8", "M": 1, "K": 4096, "N": 32000, "bias": False, "epi": "none"},
        # 32 sequences decoding together through an FFN projection.
        {"name": "i8_decode_batch32", "kind": "linear_i8", "M": 32, "K": 4096, "N": 11008, "bias": False,
         "epi": "none"},
        # A prompt chunk of 256 tokens through a square projection: few tiles for 256 CUs.
        {"name": "i8_chunk256", "kind": "linear_i8", "M": 256, "K": 4096, "N": 4096, "bias": False, "epi": "none"},
        # Nothing is a multiple of anything: a prompt of 331 tokens, the depth of the small FFN, an odd width.
        {"name": "i8_ragged", "kind": "linear_i8", "M": 331, "K": 1376, "N": 5003, "bias": True, "epi": "gelu"},
        # A prompt of 2048 tokens through a large FFN projection: the matrix cores.
        {"name": "i8_prefill", "kind": "linear_i8", "M": 2048, "K": 4096, "N": 14336, "bias": False, "epi": "none"},
        # A small f32 layer with odd sizes (a classifier or router): rows that are not 16-byte aligned.
        {"name": "f32_ragged", "kind": "linear_f32", "M": 77, "K": 1000, "N": 1001, "trans_b": 0, "bias": True,
         "epi": "silu", "beta": 0.0},
        # An f32 prefill projection, weights [N][K], bias, accumulated C and GELU.
        {"name": "f32_prefill", "kind": "linear_f32", "M": 2048, "K": 4096, "N": 4096, "trans_b": 1, "bias": True,
         "epi": "gelu", "beta": 0.5},
        # Four drafted tokens through an f32 output head stored as the embedding table is, [vocab][hidden].
        {"name": "head_tied", "kind": "head", "rows": 4, "hidden": 4096, "vocab": 32000, "trans_w": 1},
        # Causal attention over a prompt of 2048 tokens, 32 heads of 128.
        {"name": "attn_prefill", "kind": "attention", "batch": 1, "heads": 32, "seq_q": 2048, "seq_k": 2048,
         "head_dim": 128, "mask": False, "fast": False},
        # A chunk of 333 tokens behind a cache of 1168, heads of 96.
        {"name": "attn_chunk_d96", "kind": "attention", "batch": 2, "heads": 16, "seq_q": 333, "seq_k": 1501,
         "head_dim": 96, "mask": False, "fast": False},
        # One decode step of a 4096-wide layer: 8 sequences, each with 4095 cached tokens.
        {"name": "block_decode_b8", "kind": "block", "batch": 8, "tokens": 1, "past": 4095, "width": 4096,
         "heads": 32, "ffn": 11008},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _depth(rng, lo, hi):
    """A contraction depth or width: half the time a multiple of 64, else of 32, of 4, or of nothing."""
    step = rng.choice((64, 64, 64, 32, 4, 1))
    return max(step, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("linear_i8", "linear_i8", "linear_i8", "linear_f32", "linear_f32", "head", "attention",
                       "attention", "attention", "block"))
    if kind == "linear_i8":
        while True:
            M, K, N = _log_int(rng, 1, 2048), _depth(rng, 256, 11008), _depth(rng, 256, 32000)
            if M * K * N <= 2048 * 4096 * 14336:
                return {"kind": kind, "M": M, "K": K, "N": N, "bias": rng.random() < 0.5,
                        "epi": rng.choice(("none", "none", "silu", "gelu"))}
    if kind == "linear_f32":
        while True:
            M, K, N = _log_int(rng, 1, 2048), _depth(rng, 128, 8192), _depth(rng, 128, 14336)
            if M * K * N <= 2048 * 4096 * 4096:
                return {"kind": kind, "M": M, "K": K, "N": N, "trans_b": rng.randint(0, 1),
                        "bias": rng.random() < 0.7, "epi": rng.choice(("none", "silu", "gelu")),
                        "beta": rng.choice((0.0, 0.0, 0.5))}
    if kind == "head":
        while True:
            c = {"kind": kind, "rows": rng.randint(1, 8), "hidden": _log_int(rng, 512, 4096) // 64 * 64,
                 "vocab": _log_int(rng, 1000, 50000), "trans_w": rng.randint(0, 1)}
            if c["hidden"] * c["vocab"] <= 4096 * 32000:
                return c
    if kind == "attention":
        while True:
            c = {"kind": kind, "batch": rng.choice((1, 1, 2, 4, 8)), "heads": rng.choice((8, 12, 16, 32)),
                 "seq_q": rng.choice((1, 1, rng.randint(2, 4), _log_int(rng, 5, 2048), _log_int(rng, 5, 2048))),
                 "seq_k": 0, "head_dim": rng.choice((64, 64, 80, 96, 128, 128)), "mask": rng.random() < 0.2,
                 "fast": rng.random() < 0.4}
            c["seq_k"] = c["seq_q"] if c["seq_q"] > 4 and rng.random() < 0.5 else c["seq_q"] + _log_int(rng, 16, 4000)
            rows = c["batch"] * c["heads"] * c["seq_q"] * c["seq_k"]
            if (rows * c["head_dim"] <= 32 * 2048 * 1024 * 128 and rows <= (1 << 26 if c["mask"] else 1 << 40)
                    and c["batch"] * c["heads"] * c["seq_k"] * c["head_dim"] <= 8 * 32 * 4096 * 128):
                return c
    width, heads, ffn = rng.choice(((256, 4, 688), (512, 8, 1376), (1024, 8, 2752), (2048, 16, 5504),
                                    (4096, 32, 11008)))
    if rng.random() < 0.5:
        return {"kind": "block", "batch": rng.randint(1, 8), "tokens": 1, "past": _log_int(rng, 16, 2047),
                "width": width, "heads": heads, "ffn": ffn}
    return {"kind": "block", "batch": 1, "tokens": _log_int(rng, 5, 2048 if width <= 1024 else 512), "past": 0,
            "width": width, "heads": heads, "ffn": ffn}


# ---------------------------------------------------------------------------
# One device and stream for every state, and device memory that torch can see
# ---------------------------------------------------------------------------

_sessions = {}


def _session(fast=False):
    if fast not in _sessions:
        config = None
        if fast:
            config = abi.Config()
            config.abi_version = 1
            config.flags = abi.CONFIG_HIGH_THROUGHPUT
        _sessions[fast] = Session(None, config)
    return _sessions[fast]


class _Memory:
    """A vnpu buffer as torch sees it; given back when nothing refers to it."""

    TYPES = {torch.float32: ("<f4", 4), torch.int8: ("|i1", 1)}

    def __init__(self, session, shape, dtype):
        self.session = session
        typestr, size = self.TYPES[dtype]
        self.buffer = session.alloc(size * math.prod(shape))
        self.ptr = self.buffer.ptr
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (self.ptr, False),
                                         "version": 2}

    def __del__(self):
        if self.session.dev is not None:
            self.session.free(self.buffer)


def _empty(session, shape, dtype=torch.float32):
    return torch.as_tensor(_Memory(session, shape, dtype), device="cuda")


def _like(session, value):
    t = _empty(session, value.shape, value.dtype)
    t.copy_(value)
    return t


class _Packed:
    """Packed int8 weights, given back when nothing refers to them."""

    def __init__(self, session, w8, scales):
        self.session = session
        handle = C.c_void_p()
        session.check("vnpu_pack_weights_i8", session.lib.vnpu_pack_weights_i8(
            session.dev, C.c_void_p(w8.data_ptr()), C.c_void_p(scales.data_ptr()), w8.shape[0], w8.shape[1], 0, 0,
            C.byref(handle)))
        self.handle = handle

    def __del__(self):
        if self.session.dev is not None:
            self.session.lib.vnpu_packed_weights_destroy(self.handle)


def _normal(seed, tag, shape, sigma=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + sum((i + 1) * ord(ch) for i, ch in enumerate(tag)) * 7919) % (1 << 62))
    return torch.randn(tuple(shape), generator=g, device="cuda", dtype=torch.float32) * sigma


def _quantize(x, dim):
    """The int8 codes and scales of QUANTIZE_I8 (by row: dim 1, by column: dim 0), in the format's own 32 bits."""
    scale = x.abs().amax(dim=dim, keepdim=True).float() / 127.0
    inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    y = x.float() * inv
    q = torch.trunc(y + torch.copysign(torch.full_like(y, 0.5), y)).clamp(-127, 127)
    return q.to(torch.int8), scale


def _weights_i8(seed, tag, K, N):
    return _quantize(_normal(seed, tag, (K, N), 0.02), 0)


def _packets(session, *commands):
    array = (abi.Command * len(commands))()
    for i, (opcode, fields) in enumerate(commands):
        fields = {k: v.data_ptr() if isinstance(v, torch.Tensor) else v for k, v in fields.items()}
        array[i] = session.command(opcode, **fields)
    return array


class _State:
    """Packets, what they point at, and the outputs."""

    def __init__(self, session, packets, outputs, keep, after=None):
        self.session, self.packets, self.outputs, self.keep, self.after = session, packets, outputs, keep, after


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    s = state.session
    s.check("vnpu_stream_submit", s.lib.vnpu_stream_submit(s.stream, state.packets, len(state.packets), None))
    if state.after is not None:
        state.after()
    return state.outputs


def _prepare_linear_i8(c, seed):
    s = _session()
    M, K, N = c["M"], c["K"], c["N"]
    x = _like(s, _normal(seed, "x", (M, K)))
    packed = _Packed(s, *(_like(s, t) for t in _weights_i8(seed, "w", K, N)))
    bias = _like(s, _normal(seed, "bias", (N,), 0.1)) if c["bias"] else None
    a8, scale, out = _empty(s, (M, K), torch.int8), _empty(s, (M,)), _empty(s, (M, N))
    fields = {"A": a8, "B": packed.handle, "scale_a": scale, "C": out, "M": M, "K": K, "N": N,
              "epilogue": EPILOGUES[c["epi"]]}
    if bias is not None:
        fields["bias"] = bias
    packets = _packets(s, (abi.OP_QUANTIZE_I8, {"X": x, "Y": a8, "scales": scale, "rows": M, "cols": K,
                                                "axis": abi.QUANT_PER_ROW}), (abi.OP_MATMUL_I8, fields))
    return _State(s, packets, {"a8": a8, "scale": scale, "c": out}, (x, packed, bias))


def _prepare_linear_f32(c, seed):
    s = _session()
    M, K, N = c["M"], c["K"], c["N"]
    a = _like(s, _normal(seed, "a", (M, K)))
    b = _like(s, _normal(seed, "b", (N, K) if c["trans_b"] else (K, N), 0.02))
    bias = _like(s, _normal(seed, "bias", (N,), 0.1)) if c["bias"] else None
    out = _like(s, _normal(seed, "c", (M, N)))
    fields = {"A": a, "B": b, "C": out, "M": M, "K": K, "N": N, "trans_b": c["trans_b"], "alpha": 1.0,
              "beta": c["beta"], "epilogue": EPILOGUES[c["epi"]]}
    if bias is not None:
        fields["bias"] = bias
    return _State(s, _packets(s, (abi.OP_MATMUL_F32, fields)), {"c": out}, (a, b, bias))


def _prepare_head(c, seed):
    s = _session()
    g, h, v = c["rows"], c["hidden"], c["vocab"]
    hidden = _like(s, _normal(seed, "hidden", (g, h)))
    w = _like(s, _normal(seed, "w", (v, h) if c["trans_w"] else (h, v), 0.02))
    logits, probs = _empty(s, (g, v)), _empty(s, (g, v))
    packets = _packets(s, (abi.OP_MTP_HEAD_F32, {"hidden": hidden, "W": w, "logits": logits, "gamma": g,
                                                 "hidden_dim": h, "vocab": v, "trans_w": c["trans_w"]}),
                       (abi.OP_SOFTMAX_F32, {"X": logits, "Y": probs, "rows": g, "cols": v}))
    return _State(s, packets, {"logits": logits, "probs": probs}, (hidden, w))


def _attention_inputs(c, seed):
    b, h, d = c["batch"], c["heads"], c["head_dim"]
    q = _normal(seed, "q", (b, h, c["seq_q"], d))
    k = _normal(seed, "k", (b, h, c["seq_k"], d))
    v = _normal(seed, "v", (b, h, c["seq_k"], d))
    mask = None
    if c["mask"]:  # an additive bias by distance, as position biases are
        mask = -_normal(seed, "mask", (b, h, c["seq_q"], c["seq_k"]), 0.5).abs()
    return q, k, v, mask


def _prepare_attention(c, seed):
    s = _session(c["fast"])
    q, k, v, mask = (None if t is None else _like(s, t) for t in _attention_inputs(c, seed))
    o = _empty(s, q.shape)
    fields = {"Q": q, "K": k, "V": v, "O": o, "batch": c["batch"], "heads": c["heads"], "seq_q": c["seq_q"],
              "seq_k": c["seq_k"], "head_dim": c["head_dim"], "causal": 1}
    if mask is not None:
        fields["mask"] = mask
    return _State(s, _packets(s, (abi.OP_ATTENTION_F32, fields)), {"o": o}, (q, k, v, mask))


def _block_inputs(c, seed):
    d, f = c["width"], c["ffn"]
    dims = {"qkv": (d, 3 * d), "o": (d, d), "gate": (d, f), "up": (d, f), "down": (f, d)}
    w = {n: _weights_i8(seed, n, *dims[n]) for n in PROJECTIONS}
    norm = {n: 1.0 + 0.1 * _normal(seed, n, (d,)) for n in ("norm_attn", "norm_ffn")}
    x = _normal(seed, "x", (c["batch"] * c["tokens"], d))
    cache = None
    if c["past"]:
        shape = (c["batch"], c["heads"], c["past"] + c["tokens"], d // c["heads"])
        cache = _normal(seed, "k_cache", shape), _normal(seed, "v_cache", shape)
    return w, norm, x, cache


def _prepare_block(c, seed):
    s = _session()
    B, T, d, f, H = c["batch"], c["tokens"], c["width"], c["ffn"], c["heads"]
    w, norm, x, cache = _block_inputs(c, seed)
    packed = {n: _Packed(s, *(_like(s, t) for t in w[n])) for n in PROJECTIONS}
    norm = {n: _like(s, t) for n, t in norm.items()}
    x0, rows, heads = _like(s, x), B * T, (B, H, T, d // H)
    t = {n: _empty(s, shape) for n, shape in {
        "x": (rows, d), "xn": (rows, d), "scale_a": (rows,), "qkv": (rows, 3 * d), "q": heads, "k": heads, "v": heads,
        "o": heads, "att": (rows, d), "proj": (rows, d), "gate": (rows, f), "up": (rows, f), "ff": (rows, f)}.items()}
    t["a8"] = _empty(s, (rows, max(d, f)), torch.int8)
    if cache is not None:
        t["k_cache"], t["v_cache"] = _like(s, cache[0]), _like(s, cache[1])
    weights = blk.BlockWeights(*(packed[n].handle.value for n in PROJECTIONS), norm["norm_attn"].data_ptr(),
                               norm["norm_ffn"].data_ptr())
    buffers = blk.BlockBuffers(*(t[n].data_ptr() if n in t else None for n in blk.BUFFER_FIELDS))
    config = blk.BlockConfig(B, T, d, H, d // H, f, c["past"], c["past"] + T if cache is not None else 0, 1e-5, 1e4)
    table, hip, entry = s.lib.vnpu_get_backend_v1(), s.lib.vnpu_stream_hip_handle(s.stream), blk.block_lib()
    layer = (table, s.stream, hip, C.byref(config), C.byref(weights), C.byref(buffers))

    def after():
        s.check("vnpu_block_run", entry.vnpu_block_run(*layer))

    # The layer updates x in place: each pass takes its hidden states from where the layer below left them.
    packets = _packets(s, (abi.OP_COPY, {"dst": t["x"], "src": x0, "bytes": 4 * rows * d,
                                         "direction": abi.COPY_D2D}))
    kv = ("k_cache", "v_cache") if cache is not None else ("k", "v")
    return _State(s, packets, {"x": t["x"], "k": t[kv[0]], "v": t[kv[1]]}, (packed, norm, x0, t, layer), after)


# ---------------------------------------------------------------------------
# What a pass cannot do without, how close another implementation comes, and the values in 64 bits
# ---------------------------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind == "linear_i8":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 5 * M * K + 4 * M + K * N + 4 * N * (2 if c["bias"] else 1) + 4 * M * N,
                "flops": 2 * M * K * N}
    if kind == "linear_f32":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * (M * K + K * N + (N if c["bias"] else 0) + M * N * (2 if c["beta"] else 1)),
                "flops": 2 * M * K * N}
    if kind == "head":
        g, h, v = c["rows"], c["hidden"], c["vocab"]
        return {"bytes": 4 * (g * h + h * v + 2 * g * v), "flops": 2 * g * h * v}
    if kind == "attention":
        bh, sq, sk, d = c["batch"] * c["heads"], c["seq_q"], c["seq_k"], c["head_dim"]
        pairs = sq * (sk - sq) + sq * (sq + 1) // 2
        return {"bytes": 4 * bh * (2 * sq * d + 2 * sk * d + (sq * sk if c["mask"] else 0)), "flops": 4 * bh * pairs * d}
    B, T, d, f, past = c["batch"], c["tokens"], c["width"], c["ffn"], c["past"]
    params = 4 * d * d + 3 * d * f
    pairs = B * (T * past + T * (T + 1) // 2)
    return {"bytes": params + 4 * (3 * d + d + 2 * f + d + 2 * d) + 8 * B * T * d
            + 8 * B * d * (past + T), "flops": 2 * B * T * params + 4 * pairs * d}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear_i8":
        # Whole-number sums; the scales and the activation round in 32 bits.
        return {"rel": 1e-6, "max": 2e-5} if case["epi"] == "none" else {"rel": 1e-5, "max": 1e-4}
    if kind == "linear_f32":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "head":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "attention":
        return {"rel": 2e-4, "max": 2e-3} if case["fast"] else {"rel": 1e-4, "max": 1e-3}
    # A layer quantizes four times: a last-bit difference before a quantize moves codes by one.
    return {"rel": 2e-2, "max": 0.3}


def _act(y, epi):
    if epi == "silu":
        return y * torch.sigmoid(y)
    if epi == "gelu":
        return 0.5 * y * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (y + 0.044715 * y * y * y)))
    return y


def _linear_i8(x, w8, scales):
    q, s = _quantize(x, 1)
    return q, s, (q.double() @ w8.double()) * s.double() * scales.double()


def _attend(q, k, v, mask):
    """Causal attention in 64 bits; a query sees the keys up to its own place from the end."""
    sq, sk = q.shape[2], k.shape[2]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    hidden = torch.arange(sk, device=q.device)[None, :] > torch.arange(sq, device=q.device)[:, None] + (sk - sq)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            score = q[b, h].double() @ k[b, h].double().T / math.sqrt(q.shape[3])
            if mask is not None:
                score = score + mask[b, h].double()
            out[b, h] = torch.softmax(score.masked_fill(hidden, -math.inf), dim=1) @ v[b, h].double()
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "linear_i8":
        bias = _normal(seed, "bias", (c["N"],), 0.1).double() if c["bias"] else 0.0
        q, s, y = _linear_i8(_normal(seed, "x", (c["M"], c["K"])), *_weights_i8(seed, "w", c["K"], c["N"]))
        return {"a8": q, "scale": s.reshape(-1).double(), "c": _act(y + bias, c["epi"])}
    if kind == "linear_f32":
        M, K, N = c["M"], c["K"], c["N"]
        b = _normal(seed, "b", (N, K) if c["trans_b"] else (K, N), 0.02).double()
        y = _normal(seed, "a", (M, K)).double() @ (b.T if c["trans_b"] else b)
        if c["bias"]:
            y = y + _normal(seed, "bias", (N,), 0.1).double()
        return {"c": _act(y + c["beta"] * _normal(seed, "c", (M, N)).double(), c["epi"])}
    if kind == "head":
        h, v = c["hidden"], c["vocab"]
        w = _normal(seed, "w", (v, h) if c["trans_w"] else (h, v), 0.02).double()
        logits = _normal(seed, "hidden", (c["rows"], h)).double() @ (w.T if c["trans_w"] else w)
        return {"logits": logits, "probs": torch.softmax(logits, dim=1)}
    if kind == "attention":
        return {"o": _attend(*_attention_inputs(c, seed))}
    return _exact_block(c, seed)


def _exact_block(c, seed):
    w, norm, x, cache = _block_inputs(c, seed)
    B, T, d, H, past = c["batch"], c["tokens"], c["width"], c["heads"], c["past"]
    D = d // H

    def rms(y, weight):
        return y * torch.rsqrt(y.square().mean(dim=1, keepdim=True) + 1e-5) * weight.double()

    def gemm(y, name):
        return _linear_i8(y, *w[name])[2]

    def rope(y):
        inv = 1e4 ** (-torch.arange(0, D, 2, device=y.device, dtype=torch.float64) / D)
        angle = torch.arange(past, past + T, device=y.device, dtype=torch.float64)[:, None] * inv
        cos, sin, a, b = angle.cos(), angle.sin(), y[..., :D // 2], y[..., D // 2:]
        return torch.cat((a * cos - b * sin, a * sin + b * cos), dim=-1)

    x = x.double()
    q, k, v = (p.reshape(B, T, H, D).transpose(1, 2) for p in gemm(rms(x, norm["norm_attn"]), "qkv").split(d, dim=1))
    q, k = rope(q), rope(k)
    if cache is not None:
        cached = [t.double() for t in cache]
        cached[0][:, :, past:], cached[1][:, :, past:] = k, v
        k, v = cached
    x = x + gemm(_attend(q, k, v, None).transpose(1, 2).reshape(B * T, d), "o")
    y = rms(x, norm["norm_ffn"])
    x = x + gemm(_act(gemm(y, "gate"), "silu") * gemm(y, "up"), "down")
    return {"x": x, "k": k.contiguous(), "v": v.contiguous()}
