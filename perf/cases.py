"""The work that programs hand to this library, as cases that can be timed and compared.

Every case goes through the public entry points of the binding (mi355q.py, one ctypes call per
entry point of include/mi355q.h), with weights prepared once and buffers kept on the GPU as a
runtime keeps them; the hook cases hand over host arrays, because the hooks take nothing else.
Sizes are those of the models the library is written for: the 27B decoder layer (hidden 5120, MLP
17408), the 0.8B one (1024, 3584), the H3 projections (5376 -> 14336, 8-bit 5120 -> 25600), the
Whisper encoder (1280, 5120, 1500 frames) and the SenseVoice encoder (1024 -> 4096, 8-bit).
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cpu-llms-in-c_amd"))

import mi355q as engine  # noqa: E402

_TORCH = {engine.F16: torch.float16, engine.F32: torch.float32, engine.BF16: torch.bfloat16}
_BYTES = {engine.F16: 2, engine.F32: 4, engine.BF16: 2}
_META = {"f16": engine.META_F16_INTERLEAVED, "bf16": engine.META_BF16_PLANES}


def listed():
    return [
        # One token through a small model's layer: four launches of a few microseconds each.
        dict(name="decode_0p8b", kind="layer", hidden=1024, q=2048, kv=512, inter=3584, rows=1, meta="f16"),
        # One token through a layer of the 27B model: weight streaming, the library's headline.
        dict(name="decode_27b", kind="layer", hidden=5120, q=6144, kv=1024, inter=17408, rows=1, meta="bf16"),
        # A speculative batch of six tokens to be verified (depth 1 .. 7 plus one).
        dict(name="verify_27b_6", kind="layer", hidden=5120, q=6144, kv=1024, inter=17408, rows=6, meta="bf16"),
        # The vocabulary head after a decode step: the largest single stream of weights.
        dict(name="head_27b", kind="head", hidden=5120, vocab=248320, rows=1, meta="f16"),
        # Prompt chunks: the runtime cuts a prompt in chunks of 128, 64, 32 and 16 tokens and a rest.
        dict(name="chunk_27b_32", kind="layer", hidden=5120, q=6144, kv=1024, inter=17408, rows=32, meta="bf16"),
        dict(name="chunk_27b_67", kind="layer", hidden=5120, q=6144, kv=1024, inter=17408, rows=67, meta="bf16"),
        # A whole prompt at once.
        dict(name="prefill_27b_512", kind="layer", hidden=5120, q=6144, kv=1024, inter=17408, rows=512, meta="bf16"),
        # The H3 video model's projection over a clip's tokens, bf16 in and out.
        dict(name="h3_projection_4646", kind="projection", N=14336, K=5376, rows=4646, x="bf16", meta="bf16"),
        # The Whisper encoder's linears over 30 s of audio: symmetric group-128 weights, fp32 rows, bias.
        dict(name="whisper_layer_1500", kind="encoder", hidden=1280, inter=5120, rows=1500),
        # The same model's hook as its C runtime calls it, on three seconds of audio: host arrays in and out.
        dict(name="whisper_hook_150", kind="hook", N=5120, K=1280, rows=150),
        # The H3 text conditioner's 8-bit gate over a prompt.
        dict(name="h3_gate_q8_256", kind="q8", N=25600, K=5120, rows=256, meta="bf16"),
        # A SenseVoice encoder block's q, k and v on a few seconds of audio: quantize, three int8 products.
        dict(name="sensevoice_qkv_64", kind="w8a8", N=4096, K=1024, rows=64),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "head", "projection", "encoder", "hook", "q8", "w8a8"])
    meta = rng.choice(["f16", "bf16"])
    if kind == "layer":
        hidden = 64 * _spread(rng, 16, 96)
        head = 128 * rng.randint(2, 8)
        rows = rng.choice([1, rng.randint(2, 8), rng.randint(9, 128), _spread(rng, 129, 768)])
        return dict(kind=kind, hidden=hidden, q=head * rng.randint(2, 6), kv=head, inter=64 * _spread(rng, 56, 272),
                    rows=rows, meta=meta)
    if kind == "head":
        return dict(kind=kind, hidden=64 * _spread(rng, 16, 80), vocab=_spread(rng, 32000, 248320),
                    rows=rng.choice([1, 1, rng.randint(2, 8)]), meta=meta)
    if kind == "projection":
        return dict(kind=kind, N=_spread(rng, 2048, 14336), K=64 * _spread(rng, 32, 84), rows=_spread(rng, 11, 4646),
                    x=rng.choice(["bf16", "f16"]), meta=meta)
    if kind == "encoder":
        hidden = 128 * _spread(rng, 4, 12)
        return dict(kind=kind, hidden=hidden, inter=4 * hidden, rows=_spread(rng, 50, 1500))
    if kind == "hook":
        return dict(kind=kind, N=_spread(rng, 512, 5120), K=128 * _spread(rng, 6, 40), rows=_spread(rng, 1, 1500))
    if kind == "q8":
        return dict(kind=kind, N=_spread(rng, 4096, 25600), K=64 * _spread(rng, 24, 80), rows=_spread(rng, 1, 640),
                    meta=meta)
    return dict(kind=kind, N=_spread(rng, 512, 4096), K=16 * _spread(rng, 32, 128), rows=_spread(rng, 11, 768))


# ---- weights, quantized on the GPU from a seed's normal matrix ---------------------------------


@functools.lru_cache(maxsize=None)
def _context():
    """The program's one context (one stream, one set of staging buffers)."""
    return engine.Context(0)


class _Prepared:
    """A prepared weight that is given back with the state that holds it."""

    def __init__(self, handle, N, K, destroy):
        self.handle, self.N, self.K, self._destroy = handle, N, K, destroy

    def __del__(self):
        self._destroy(self.handle)


def _pointer(tensor):
    return ctypes.c_void_p(tensor.data_ptr())


def _row_blocks(N, K):
    step = max(1, (1 << 26) // K)
    return [(low, min(N, low + step)) for low in range(0, N, step)]


def _affine_planes(generator, N, K, meta, bits):
    """Min/max affine codes of N(0, 0.02) rows per 64 columns, and their scales and biases."""
    top = (1 << bits) - 1
    codes = torch.empty((N, K * bits // 8), dtype=torch.uint8, device="cuda")
    scales = torch.empty((N, K // 64), dtype=torch.float16 if meta == "f16" else torch.bfloat16, device="cuda")
    biases = torch.empty_like(scales)
    for low, high in _row_blocks(N, K):
        w = torch.randn((high - low, K // 64, 64), device="cuda", generator=generator).mul_(0.02)
        smallest, largest = torch.aminmax(w, dim=2)
        scales[low:high], biases[low:high] = (largest - smallest) / top, smallest
        scale, bias = scales[low:high].float().unsqueeze(2), biases[low:high].float().unsqueeze(2)
        q = w.sub_(bias).div_(scale).round_().clamp_(0, top).to(torch.uint8).view(high - low, K)
        codes[low:high] = q if bits == 8 else q[:, 0::2] | (q[:, 1::2] << 4)
    if meta == "f16":
        return codes, torch.stack((scales, biases), dim=2).contiguous(), None
    return codes, scales, biases


def _affine_q4(generator, N, K, meta):
    codes, a, b = _affine_planes(generator, N, K, meta, 4)
    torch.cuda.synchronize()
    made = _context().q4_prepare(_pointer(codes), _pointer(a), None if b is None else _pointer(b), N, K, _META[meta],
                                 engine.SOURCE_DEVICE)
    return _Prepared(made.handle, N, K, engine.library().mi355q_q4_weight_destroy)


def _affine_q8(generator, N, K, meta):
    codes, a, b = (None if t is None else t.cpu().view(torch.uint8).numpy()
                   for t in _affine_planes(generator, N, K, meta, 8))
    return _Prepared(_context().q8_prepare(codes, a, b, N, K, _META[meta]), N, K,
                     engine.library().mi355q_q8_weight_destroy)


def _sym128_records(generator, N, K):
    """[N][K/128] records: a bf16 scale, then 64 bytes of two's complement nibbles."""
    w = torch.randn((N, K // 128, 128), device="cuda", generator=generator).mul_(0.02)
    scale = (w.abs().amax(dim=2) / 7).to(torch.bfloat16)
    q = (w / scale.float().unsqueeze(2)).round_().clamp_(-8, 7).to(torch.int8).view(torch.uint8) & 15
    records = torch.empty((N, K // 128, 66), dtype=torch.uint8, device="cuda")
    records[:, :, :2] = scale.unsqueeze(2).view(torch.uint8)
    records[:, :, 2:] = q[:, :, 0::2] | (q[:, :, 1::2] << 4)
    return records


def _sym128(generator, N, K):
    records = _sym128_records(generator, N, K)
    torch.cuda.synchronize()
    made = _context().sym128_prepare(_pointer(records), N, K, engine.SYM128_ROW_MAJOR, engine.SOURCE_DEVICE)
    return _Prepared(made.handle, N, K, engine.library().mi355q_q4_weight_destroy)


def _int8_rows(generator, N, K):
    w = torch.randn((N, K), device="cuda", generator=generator).mul_(0.02)
    scale = w.abs().amax(dim=1, keepdim=True) / 127
    q = (w / scale).round_().clamp_(-127, 127).to(torch.int8)
    rows = torch.cat((scale.view(torch.uint8), q.view(torch.uint8)), dim=1).contiguous().cpu().numpy()
    return _Prepared(_context().w8a8_prepare(rows, N, K), N, K, engine.library().mi355q_w8a8_weight_destroy)


def _normal(generator, shape, dtype=engine.F16, sigma=1.0):
    return torch.randn(shape, device="cuda", generator=generator).mul_(sigma).to(_TORCH[dtype])


def _empty(shape, dtype=engine.F16):
    return torch.empty(shape, dtype=_TORCH[dtype], device="cuda")


# ---- the calls a state keeps ----------------------------------------------------------------


def _call(x, x_dtype, y_dtype, targets, residual_dtype=engine.F32, flags=0):
    """One (multi-)linear of a sequence: targets are (weight, y[, residual]) with tensors."""
    pointers = [tuple([t[0]] + [None if v is None else v.data_ptr() for v in t[1:]]) for t in targets]
    return pointers, x.data_ptr(), x_dtype, x.shape[0], y_dtype, residual_dtype, flags


def _prepare_layer(c, g):
    """A decoder layer's seven linears.  Up to 16 rows gate and up are one fused call whose output
    the down projection reads; above, the activation between them is the caller's own kernel."""
    M, H, I = c["rows"], c["hidden"], c["inter"]
    shapes = dict(q=(c["q"], H), k=(c["kv"], H), v=(c["kv"], H), o=(H, c["q"]), gate=(I, H), up=(I, H), down=(H, I))
    w = {name: _affine_q4(g, N, K, c["meta"]) for name, (N, K) in shapes.items()}
    x, attended, x_mlp = _normal(g, (M, H)), _normal(g, (M, c["q"])), _normal(g, (M, H))
    stream = _normal(g, (M, H), engine.F32)
    y = {name: _empty((M, shapes[name][0])) for name in ("q", "k", "v")}
    y["o"], y["down"] = _empty((M, H), engine.F32), _empty((M, H), engine.F32)
    calls = [_call(x, engine.F16, engine.F16, [(w[n], y[n]) for n in ("q", "k", "v")]),
             _call(attended, engine.F16, engine.F32, [(w["o"], y["o"], stream)])]
    if M <= 16:
        between = y["h"] = _empty((M, I))
        calls.append(_call(x_mlp, engine.F16, engine.F16, [(w["gate"], between), (w["up"], None)],
                           flags=engine.FUSE_GATE_UP_SILU))
    else:
        between = _normal(g, (M, I))
        y["gate"], y["up"] = _empty((M, I)), _empty((M, I))
        calls.append(_call(x_mlp, engine.F16, engine.F16, [(w["gate"], y["gate"]), (w["up"], y["up"])]))
    calls.append(_call(between, engine.F16, engine.F32, [(w["down"], y["down"], stream)]))
    return dict(calls=calls, out=y, keep=(w, x, attended, x_mlp, stream, between))


def _prepare_head(c, g):
    w, x = _affine_q4(g, c["vocab"], c["hidden"], c["meta"]), _normal(g, (c["rows"], c["hidden"]))
    y = _empty((c["rows"], c["vocab"]), engine.F32)
    return dict(calls=[_call(x, engine.F16, engine.F32, [(w, y)])], out=y, keep=(w, x))


def _prepare_projection(c, g):
    dtype = engine.BF16 if c["x"] == "bf16" else engine.F16
    w, x = _affine_q4(g, c["N"], c["K"], c["meta"]), _normal(g, (c["rows"], c["K"]), dtype)
    y = _empty((c["rows"], c["N"]), dtype)
    return dict(calls=[_call(x, dtype, dtype, [(w, y)])], out=y, keep=(w, x))


def _prepare_encoder(c, g):
    """An encoder layer's six linears with their biases, everything fp32."""
    M, H, I = c["rows"], c["hidden"], c["inter"]
    shapes = dict(q=(H, H), k=(H, H), v=(H, H), o=(H, H), fc1=(I, H), fc2=(H, I))
    w = {name: _sym128(g, N, K) for name, (N, K) in shapes.items()}
    b = {name: _normal(g, (N,), engine.F32, 0.1) for name, (N, K) in shapes.items()}
    y = {name: _empty((M, N), engine.F32) for name, (N, K) in shapes.items()}
    x = {name: _normal(g, (M, K), engine.F32) for name, K in (("qkv", H), ("o", H), ("fc1", H), ("fc2", I))}
    calls = [_call(x["qkv"], engine.F32, engine.F32, [(w[n], y[n], b[n]) for n in ("q", "k", "v")],
                   flags=engine.RESIDUAL_IS_BIAS)]
    calls += [_call(x[n], engine.F32, engine.F32, [(w[n], y[n], b[n])], flags=engine.RESIDUAL_IS_BIAS)
              for n in ("o", "fc1", "fc2")]
    return dict(calls=calls, out=y, keep=(w, b, x))


_mapped = []  # records the hooks have seen: mapped for the life of the process, as an image file is


def _prepare_hook(c, g):
    records = _sym128_records(g, c["N"], c["K"]).cpu().numpy().reshape(-1)
    _mapped.append(records)
    x = _normal(g, (c["rows"], c["K"]), engine.F32).cpu().numpy()
    bias = _normal(g, (c["N"],), engine.F32, 0.1).cpu().numpy()
    state = dict(records=records, x=x, bias=bias, N=c["N"])
    engine.hook_q4_gemm(records, x[:1], c["N"], bias)  # the first sight of a tensor uploads it
    return state


def _prepare_q8(c, g):
    w, x = _affine_q8(g, c["N"], c["K"], c["meta"]), _normal(g, (c["rows"], c["K"]))
    return dict(w=w, x=x, y=_empty((c["rows"], c["N"])))


def _prepare_w8a8(c, g):
    M, N, K = c["rows"], c["N"], c["K"]
    w = [_int8_rows(g, N, K) for _ in range(3)]
    return dict(w=w, x=_normal(g, (M, K), engine.F32), bias=[_normal(g, (N,), engine.F32, 0.1) for _ in w],
                q=torch.empty((M, K), dtype=torch.int8, device="cuda"), scales=_empty((M,), engine.F32),
                y=[_empty((M, N), engine.F32) for _ in w])


_PREPARE = dict(layer=_prepare_layer, head=_prepare_head, projection=_prepare_projection, encoder=_prepare_encoder,
                hook=_prepare_hook, q8=_prepare_q8, w8a8=_prepare_w8a8)


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, _generator(seed))
    state["kind"] = case["kind"]
    if "calls" in state:
        state["calls"] = engine.make_calls(state["calls"])
    torch.cuda.synchronize()
    return state


def run(state):
    kind = state["kind"]
    if kind == "hook":
        return engine.hook_q4_gemm(state["records"], state["x"], state["N"], state["bias"])
    ctx = _context()
    if kind == "q8":
        x, y = state["x"], state["y"]
        ctx.q8_linear_device(state["w"].handle, x.data_ptr(), engine.F16, x.shape[0], y.data_ptr(), engine.F16)
        return y
    if kind == "w8a8":
        x, q, scales = state["x"], state["q"], state["scales"]
        M, K = x.shape
        ctx.quantize_i8_device(x.data_ptr(), M, K, q.data_ptr(), scales.data_ptr())
        ctx.w8a8_linear_multi_device([w.handle for w in state["w"]], q.data_ptr(), scales.data_ptr(), M,
                                     [b.data_ptr() for b in state["bias"]], [y.data_ptr() for y in state["y"]])
        return dict(q=q, scales=scales, y=state["y"])
    ctx.q4_sequence(state["calls"])
    return state["out"]


# ---- the same in 64 bits, from the codes a state was made of -----------------------------------


def _generator(seed):
    generator = torch.Generator(device="cuda")
    generator.manual_seed(int(seed))
    return generator


def _product64(x, N, K, values):
    """x [M][K] times the transpose of a weight whose rows low .. high values(low, high) gives."""
    y = torch.empty((x.shape[0], N), dtype=torch.float64, device="cuda")
    for low, high in _row_blocks(N, K):
        y[:, low:high] = x.double() @ values(low, high).t()
    return y


def _affine64(generator, N, K, meta, bits=4):
    """A function of x: the product with the weight that _affine_planes draws here."""
    codes, a, b = _affine_planes(generator, N, K, meta, bits)

    def values(low, high):
        q = codes[low:high]
        q = q if bits == 8 else torch.stack((q & 15, q >> 4), dim=2)
        scale, bias = (a[low:high, :, 0], a[low:high, :, 1]) if b is None else (a[low:high], b[low:high])
        q = q.reshape(high - low, K // 64, 64).double()
        return q.mul_(scale.double().unsqueeze(2)).add_(bias.double().unsqueeze(2)).view(high - low, K)

    return lambda x: _product64(x, N, K, values)


def _sym64(generator, N, K):
    records = _sym128_records(generator, N, K)

    def values(low, high):
        scale = records[low:high, :, :2].contiguous().view(torch.bfloat16).double()
        q = records[low:high, :, 2:]
        q = torch.stack((q & 15, q >> 4), dim=3).view(high - low, K // 128, 128).double()
        return torch.where(q < 8, q, q - 16).mul_(scale).view(high - low, K)

    return lambda x: _product64(x, N, K, values)


def _exact_layer(c, g):
    M, H, I = c["rows"], c["hidden"], c["inter"]
    shapes = dict(q=(c["q"], H), k=(c["kv"], H), v=(c["kv"], H), o=(H, c["q"]), gate=(I, H), up=(I, H), down=(H, I))
    w = {name: _affine64(g, N, K, c["meta"]) for name, (N, K) in shapes.items()}
    x, attended, x_mlp = _normal(g, (M, H)), _normal(g, (M, c["q"])), _normal(g, (M, H))
    stream = _normal(g, (M, H), engine.F32).double()
    y = {name: w[name](x) for name in ("q", "k", "v")}
    y["o"] = w["o"](attended) + stream
    gate, up = w["gate"](x_mlp), w["up"](x_mlp)
    if M <= 16:
        y["h"] = torch.nn.functional.silu(gate) * up
        between = y["h"].half()  # an fp16 buffer between the two calls
    else:
        y["gate"], y["up"] = gate, up
        between = _normal(g, (M, I))
    y["down"] = w["down"](between) + stream
    return y


def _exact_encoder(c, g):
    M, H, I = c["rows"], c["hidden"], c["inter"]
    shapes = dict(q=(H, H), k=(H, H), v=(H, H), o=(H, H), fc1=(I, H), fc2=(H, I))
    w = {name: _sym64(g, N, K) for name, (N, K) in shapes.items()}
    b = {name: _normal(g, (N,), engine.F32, 0.1) for name, (N, K) in shapes.items()}
    x = {name: _normal(g, (M, K), engine.F32) for name, K in (("qkv", H), ("o", H), ("fc1", H), ("fc2", I))}
    return {name: w[name](x["qkv" if name in "qkv" else name]) + b[name].double() for name in shapes}


def _exact_w8a8(c, g):
    M, N, K = c["rows"], c["N"], c["K"]
    weights = []
    for _ in range(3):
        w = torch.randn((N, K), device="cuda", generator=g).mul_(0.02)
        scale = w.abs().amax(dim=1, keepdim=True) / 127
        weights.append(((w / scale).round_().clamp_(-127, 127).double(), scale.double()))
    x = _normal(g, (M, K), engine.F32)
    bias = [_normal(g, (N,), engine.F32, 0.1) for _ in weights]
    scales = x.abs().amax(dim=1) / 127
    q = (x * (1 / scales).unsqueeze(1)).round_().double()
    y = [(q @ w.t()) * scale.t() * scales.double().unsqueeze(1) + b.double() for (w, scale), b in zip(weights, bias)]
    return dict(q=None, scales=x.abs().amax(dim=1).double() / 127, y=y)


def exact(case, seed):
    """What run() returns for these inputs, in 64 bits and with the weights' exact values."""
    c, g = case, _generator(seed)
    if c["kind"] == "layer":
        return _exact_layer(c, g)
    if c["kind"] == "encoder":
        return _exact_encoder(c, g)
    if c["kind"] == "w8a8":
        return _exact_w8a8(c, g)
    if c["kind"] == "hook":
        weight = _sym64(g, c["N"], c["K"])
        x, bias = _normal(g, (c["rows"], c["K"]), engine.F32), _normal(g, (c["N"],), engine.F32, 0.1)
        return weight(x) + bias.double()
    if c["kind"] == "head":
        return _affine64(g, c["vocab"], c["hidden"], c["meta"])(_normal(g, (c["rows"], c["hidden"])))
    weight = _affine64(g, c["N"], c["K"], c["meta"], 8 if c["kind"] == "q8" else 4)
    return weight(_normal(g, (c["rows"], c["K"]), engine.BF16 if c.get("x") == "bf16" else engine.F16))


# ---- what a pass cannot do without ----------------------------------------------------------


def _q4_bytes(N, K):
    return N * K // 2 + N * (K // 64) * 4


def work(case):
    c, M = case, case["rows"]
    if c["kind"] == "layer":
        H, Q, V, I = c["hidden"], c["q"], c["kv"], c["inter"]
        weights = _q4_bytes(Q + 2 * V, H) + _q4_bytes(H, Q) + _q4_bytes(2 * I, H) + _q4_bytes(H, I)
        # x of q|k|v, of o and of gate|up; the outputs; the residual rows of o and down
        cells = 2 * (2 * H + Q) + 2 * (Q + 2 * V) + 4 * 4 * H
        cells += 2 * I if M <= 16 else 2 * I + 2 * 2 * I  # h, or down's x and gate's and up's outputs
        return dict(bytes=weights + M * cells, flops=2 * M * (H * (Q + 2 * V) + H * Q + 3 * H * I))
    if c["kind"] == "encoder":
        H, I = c["hidden"], c["inter"]
        pairs = 4 * H * H + 2 * H * I
        return dict(bytes=pairs // 2 + pairs // 64 + 4 * (5 * H + I) + 4 * M * (3 * H + I + 5 * H + I), flops=2 * M * pairs)
    if c["kind"] == "hook":
        N, K = c["N"], c["K"]
        return dict(bytes=N * K // 2 + N * (K // 128) * 2 + 4 * N + 4 * M * (N + K), flops=2 * M * N * K)
    if c["kind"] == "w8a8":
        N, K = c["N"], c["K"]
        return dict(bytes=3 * N * (K + 8) + M * (5 * K + 4) + 4 * 3 * M * N, flops=2 * 3 * M * N * K)
    if c["kind"] == "q8":
        N, K = c["N"], c["K"]
        return dict(bytes=N * K + N * (K // 64) * 4 + 2 * M * (N + K), flops=2 * M * N * K)
    N, K = (c["vocab"], c["hidden"]) if c["kind"] == "head" else (c["N"], c["K"])
    return dict(bytes=_q4_bytes(N, K) + 2 * M * K + (4 if c["kind"] == "head" else 2) * M * N, flops=2 * M * N * K)


def tolerance(case):
    kind = case["kind"]
    if kind == "w8a8":
        return "exact"  # integer sums, and one fixed order of fp32 operations behind them
    if kind in ("encoder", "hook"):
        return dict(rel=2e-6)  # fp32 rows, weights of eleven bits: the sums' own rounding
    if kind == "projection" and case["x"] == "bf16":
        return dict(rel=6e-3)  # one rounding to bf16
    return dict(rel=1e-3)  # one rounding to fp16, of the output or (above 16 rows) of the weight
