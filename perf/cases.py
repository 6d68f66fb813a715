"""The work a user of this library has it do, case by case, for timing and for
comparing outputs: decoding with one vector, decoding a small batch, running a
prompt through the projections, and preparing weights when a model is loaded.

Sizes come from this repository's configurations (python/wxo_workloads.py): the
2048 / 5632 decoder layer, the 11008 x 4096 projection, the ragged 4096 x 4099
one and the 151936 x 1024 vocabulary head.  Every case goes through the Python
binding's device-pointer entry points, on torch tensors that stay on the GPU.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "web-xpu-ops_amd", "python"))
import wxo_q8  # noqa: E402

DEVICE = "cuda"
HIDDEN, FFN = 2048, 5632
LAYERS = 4  # of one decode step: their 205 MB of weights pass through the caches once a step


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # Decoding one token, one projection alone: the smallest call there is.
        {"name": "decode_2048x2048", "kind": "matvec", "N": 2048, "K": 2048, "M": 1},
        # Decoding one token at the larger projection.
        {"name": "decode_11008x4096", "kind": "matvec", "N": 11008, "K": 4096, "M": 1},
        # Rows that are no multiple of 16 bytes.
        {"name": "decode_4096x4099", "kind": "matvec", "N": 4096, "K": 4099, "M": 1},
        # One decode step's projections of several layers, replayed as a HIP graph:
        # q/k/v in one launch, o and down with their residual, gate/up fused.
        {"name": "decode_step", "kind": "decode_step", "hidden": HIDDEN, "ffn": FFN, "layers": LAYERS},
        # A batch of 16 sequences decoding together, one projection.
        {"name": "batch16_11008x4096", "kind": "matvec", "N": 11008, "K": 4096, "M": 16},
        # A batch of 8 at the vocabulary head.
        {"name": "batch8_head", "kind": "matvec", "N": 151936, "K": 1024, "M": 8},
        # A prompt of a sentence: gate and up on the same activations.
        {"name": "prompt24_gate_up", "kind": "prompt", "tokens": 24, "N": FFN, "K": HIDDEN, "count": 2},
        # A prompt of a paragraph, its length no multiple of any tile: q, k and v.
        {"name": "prompt77_qkv", "kind": "prompt", "tokens": 77, "N": HIDDEN, "K": HIDDEN, "count": 3},
        # A prompt of a page: gate and up.
        {"name": "prompt512_gate_up", "kind": "prompt", "tokens": 512, "N": FFN, "K": HIDDEN, "count": 2},
        # A long prompt: down, whose activations are the gated product.
        {"name": "prompt2048_down", "kind": "prompt", "tokens": 2048, "N": HIDDEN, "K": FFN, "count": 1, "gated": True},
        # Loading f32 weights: quantize and pack one matrix.
        {"name": "load_quantize_pack", "kind": "quantize_pack", "N": FFN, "K": HIDDEN},
        # Loading int8 codes with ragged rows.
        {"name": "load_pack_int8_4096x4099", "kind": "pack_int8", "N": 4096, "K": 4099},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A row length or row count: mostly multiples of 64, as model dimensions
    are, sometimes any number."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.3 else max(lo, n // 64 * 64)


def draw(rng):
    kind = rng.choice(["matvec", "batch", "batch", "head", "prompt", "prompt", "prompt", "decode_step",
                       "quantize_pack", "pack_int8"])
    if kind == "matvec":
        return {"kind": "matvec", "N": _width(rng, 512, 12288), "K": _width(rng, 512, 12288), "M": 1}
    if kind == "batch":
        return {"kind": "matvec", "N": _width(rng, 1024, 12288), "K": _width(rng, 1024, 12288), "M": _log_int(rng, 2, 32)}
    if kind == "head":
        return {"kind": "matvec", "N": _width(rng, 16384, 151936), "K": 64 * rng.randint(8, 16), "M": rng.randint(1, 16)}
    if kind == "prompt":
        while True:
            c = {"kind": "prompt", "tokens": _log_int(rng, 4, 2048), "N": _width(rng, 1024, 8192),
                 "K": _width(rng, 1024, 8192), "count": rng.randint(1, 3), "gated": rng.random() < 0.3}
            if c["tokens"] * c["N"] * c["K"] * c["count"] <= 2048 * HIDDEN * FFN:
                return c
    if kind == "decode_step":
        hidden = 64 * rng.randint(16, 32)
        return {"kind": "decode_step", "hidden": hidden, "ffn": _width(rng, 2 * hidden, 2 * hidden + 1536),
                "layers": rng.randint(1, LAYERS)}
    return {"kind": kind, "N": _width(rng, 512, 8192), "K": _width(rng, 512, 8192)}


# ------------------------------------------------------------------ inputs

def _words(K):
    return (K + 3) // 4


def _quantized(gen, N, K):
    """Per-row absmax int8 of N(0, 0.02) weights, in the wire format: packed
    words as an int32 tensor [N, ceil(K/4)] and scales f32 [N]."""
    w = torch.randn(N, K, generator=gen, device=DEVICE, dtype=torch.float32) * 0.02
    scale = w.abs().amax(dim=1) / 127.0
    codes = torch.zeros(N, 4 * _words(K), dtype=torch.int8, device=DEVICE)
    codes[:, :K] = torch.round(w / scale[:, None]).clamp_(-127, 127).to(torch.int8)
    return codes.view(torch.int32), scale


def _activations(gen, rows, K, gated=False):
    """N(0, 1), as after a norm, or silu(g) * u of two such, as before down."""
    x = torch.randn(rows, K, generator=gen, device=DEVICE, dtype=torch.float32)
    if gated:
        x = torch.nn.functional.silu(x) * torch.randn(rows, K, generator=gen, device=DEVICE, dtype=torch.float32)
    return x


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEVICE)


def _inputs(case, seed):
    """The tensors a pass reads, made from the seed alone."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    kind = case["kind"]
    if kind == "matvec":
        weight, scale = _quantized(gen, case["N"], case["K"])
        return {"weight": weight, "scale": scale, "x": _activations(gen, case["M"], case["K"])}
    if kind == "prompt":
        weights = [_quantized(gen, case["N"], case["K"]) for _ in range(case["count"])]
        return {"weights": weights, "a": _activations(gen, case["tokens"], case["K"], case.get("gated", False))}
    if kind == "decode_step":
        h, f = case["hidden"], case["ffn"]
        shapes = {"q": (h, h), "k": (h, h), "v": (h, h), "o": (h, h), "gate": (f, h), "up": (f, h), "down": (h, f)}
        layers = [{name: _quantized(gen, *shape) for name, shape in shapes.items()} for _ in range(case["layers"])]
        return {"layers": layers, "x": _activations(gen, 1, h), "attended": _activations(gen, case["layers"], h)}
    if kind == "quantize_pack":
        w = torch.randn(case["N"], case["K"], generator=gen, device=DEVICE, dtype=torch.float32) * 0.02
        return {"w": w}
    if kind == "pack_int8":
        codes = torch.randint(-127, 128, (case["N"], case["K"]), generator=gen, device=DEVICE, dtype=torch.int8)
        return {"codes": codes}
    raise ValueError(kind)


def _ptr(t):
    return t.data_ptr()


def _record_decode_step(s, h, f, stream):
    """The projections of one decode step in the resident engine's order.  The
    attention and the norms between them are other programs' work: `attended`
    stands for their result, and each layer reads the residual stream as it is."""
    x = _ptr(s["x"])
    for i, layer in enumerate(s["layers"]):
        def w(name):
            return [_ptr(t) for t in layer[name]]
        out = s["buffers"][i]
        wxo_q8.matvec_q8_multi_device([(*w(n), _ptr(out[n]), h) for n in ("q", "k", "v")], x, h, stream=stream)
        wxo_q8.matvec_q8_residual_device(*w("o"), _ptr(s["attended"][i]), x, _ptr(out["o"]), h, h, stream=stream)
        wxo_q8.matvec_q8_ffn_device(*w("gate"), *w("up"), _ptr(out["o"]), _ptr(out["ffn"]), f, h, stream=stream)
        wxo_q8.matvec_q8_residual_device(*w("down"), _ptr(out["ffn"]), _ptr(out["o"]), _ptr(out["down"]), h, f,
                                         stream=stream)
        x = _ptr(out["down"])


def prepare(case, seed):
    wxo_q8.init()
    s = {"case": dict(case), **_inputs(case, seed)}
    kind = case["kind"]
    if kind == "matvec":
        s["y"] = _empty(case["M"], case["N"])
    elif kind == "prompt":
        s["y"] = [_empty(case["tokens"], case["N"]) for _ in range(case["count"])]
        s["workspace_bytes"] = wxo_q8.matmul_q8_workspace_bytes()
        s["workspace"] = _empty(s["workspace_bytes"], dtype=torch.uint8)
    elif kind == "decode_step":
        h, f = case["hidden"], case["ffn"]
        s["buffers"] = [{n: _empty(f if n == "ffn" else h) for n in ("q", "k", "v", "o", "ffn", "down")}
                        for _ in range(case["layers"])]
        torch.cuda.synchronize()
        s["stream"] = wxo_q8.Stream()
        s["graph"] = wxo_q8.Graph.capture(s["stream"], lambda: _record_decode_step(s, h, f, s["stream"]))
    elif kind == "quantize_pack":
        s["packed"] = _empty(case["N"], _words(case["K"]), dtype=torch.int32)
        s["scale"] = _empty(case["N"])
    elif kind == "pack_int8":
        s["packed"] = _empty(case["N"], _words(case["K"]), dtype=torch.int32)
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "matvec":
        wxo_q8.matvec_q8_device(_ptr(s["weight"]), _ptr(s["scale"]), _ptr(s["x"]), _ptr(s["y"]), c["N"], c["K"], c["M"])
        return s["y"]
    if kind == "prompt":
        wxo_q8.matmul_q8_multi_device(
            _ptr(s["a"]), [(_ptr(w), _ptr(sc), _ptr(y), c["N"]) for (w, sc), y in zip(s["weights"], s["y"])],
            c["tokens"], c["K"], workspace=_ptr(s["workspace"]), workspace_bytes=s["workspace_bytes"])
        return s["y"]
    if kind == "decode_step":
        s["graph"].launch(s["stream"])
        return s["buffers"]
    if kind == "quantize_pack":
        wxo_q8.quantize_pack_q8_device(_ptr(s["w"]), c["N"], c["K"], _ptr(s["packed"]), _ptr(s["scale"]))
        return {"packed": s["packed"], "scale": s["scale"]}
    if kind == "pack_int8":
        wxo_q8.pack_int8_rows_device(_ptr(s["codes"]), c["N"], c["K"], _ptr(s["packed"]))
        return s["packed"]
    raise ValueError(kind)


# ------------------------------------------------------------------ what a pass cannot do without

def _projection(N, K, M):
    """Bytes and operations of one packed weight against M vectors, without the vectors."""
    return 4 * N * _words(K) + 4 * N + 4 * N * M, 2 * N * K * M


def work(case):
    kind = case["kind"]
    if kind in ("matvec", "prompt"):
        M, N, K, count = case.get("M") or case["tokens"], case["N"], case["K"], case.get("count", 1)
        b, f = _projection(N, K, M)
        return {"bytes": count * b + 4 * K * M, "flops": count * f}
    if kind == "decode_step":
        h, f = case["hidden"], case["ffn"]
        parts = [_projection(h, h, 1)] * 4 + [_projection(f, h, 1)] * 2 + [_projection(h, f, 1)]
        # vectors read: x, the attended one, two residuals, o's and the gated product; gate and up leave one vector
        layer = sum(p[0] for p in parts) + 4 * (5 * h + f) - 4 * f
        return {"bytes": case["layers"] * layer, "flops": case["layers"] * sum(p[1] for p in parts)}
    N, K = case["N"], case["K"]
    if kind == "quantize_pack":
        return {"bytes": 4 * N * K + 4 * N * _words(K) + 4 * N, "flops": 2 * N * K}
    return {"bytes": N * K + 4 * N * _words(K), "flops": 0}


def tolerance(case):
    """Packed words and scales are exact.  Sums are taken in 32 bits over up to
    12288 products in an order that is the kernel's own; against 64 bits the
    calls measure 0.7e-7 to 3.2e-7, a decode step of four layers up to 4e-7."""
    if case["kind"] in ("quantize_pack", "pack_int8"):
        return "exact"
    return {"rel": 1.5e-6, "max": 1.5e-5}


# ------------------------------------------------------------------ the same in 64 bits

def _dequantized(weight, scale, K):
    N = weight.shape[0]
    codes = weight.view(torch.int8).reshape(N, -1)[:, :K]
    return codes.to(torch.float64) * scale.to(torch.float64)[:, None]


def exact(case, seed):
    s = _inputs(case, seed)
    kind, K = case["kind"], case.get("K")
    if kind == "matvec":
        return s["x"].double() @ _dequantized(s["weight"], s["scale"], K).t().contiguous()
    if kind == "prompt":
        a = s["a"].double()
        return [a @ _dequantized(w, sc, K).t().contiguous() for w, sc in s["weights"]]
    if kind == "decode_step":
        h, f = case["hidden"], case["ffn"]
        outs, x = [], s["x"].reshape(-1).double()
        for i, layer in enumerate(s["layers"]):
            def mv(name, v):
                return _dequantized(*layer[name], v.numel()) @ v
            out = {n: mv(n, x) for n in ("q", "k", "v")}
            out["o"] = x + mv("o", s["attended"][i].double())
            out["ffn"] = torch.nn.functional.silu(mv("gate", out["o"])) * mv("up", out["o"])
            out["down"] = out["o"] + mv("down", out["ffn"])
            outs.append(out)
            x = out["down"]
        return outs
    if kind == "quantize_pack":
        # the scale is one f64 quotient rounded to f32, checked here; the codes
        # are whole numbers and compared as they are
        return {"packed": None, "scale": s["w"].abs().amax(dim=1).double() / 127.0}
    return None
