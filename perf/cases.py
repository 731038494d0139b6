"""What the MoE block is timed on.

Each case is work that a program using the library has it do, through the
Python binding of the C ABI: one layer or a whole stack of a decode step, one
layer of a prompt, and the weight converter.  Weights have the sizes of the
model (2048 wide, 256 experts of 512, top 8, a shared expert of 512); their
values are random, with the spread of trained ones (a weight's rms is 0.02), so
that the residual stream stays in the range a model has.  `bias` is the router
bias: 0 means none (every expert equally likely), s > 0 means log Zipf(s)
popularity over a random order of the experts, as the benchmark has it.

  kind "layer":   one call on one layer, T tokens.  entry "normed" takes
                  normalised input and adds no residual, "forward" is the layer's
                  whole MoE section (norm, MoE, residual), "norm" also writes the
                  next block's normalised input.
  kind "stack":   one call over `layers` layers, T tokens (a decode step).
  kind "rows":    rows of weights quantised to IQ4_NL rows.
  kind "convert": a layer's routed experts quantised into the arena.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qe-qwen36-b50_amd"))
import qe_moe  # noqa: E402

D, E, K, FF = 2048, 256, 8, 512
BLK = 32
EPS = 1e-6
GU_ROW, DN_ROW = D // 2 + D // BLK * 2, FF // 2 + FF // BLK * 2  # bytes of an IQ4_NL row
DOWN = 2 * FF * GU_ROW  # an expert's down rows start here
EXPERT = DOWN + D * DN_ROW
DENSE = 1024 * (D + D // BLK * 2) + D * (FF + FF // BLK * 2) + 257 * D * 4 + D * 4  # shared expert, router, norm
FLOP_TOKEN = (K + 1) * 6 * D * FF + 2 * 257 * D
CODEBOOK = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
SOURCES = {"f32": (qe_moe.SRC_F32, 128), "f16": (qe_moe.SRC_F16, 64), "bf16": (qe_moe.SRC_BF16, 64),
           "q8_0": (qe_moe.SRC_Q8_0, 34)}  # ggml type id, bytes of a 32-block


def listed():
    return [
        # one layer of a one-token decode step, as an engine that runs its own
        # attention between the layers calls it: the smallest call there is
        {"name": "decode_1_layer", "kind": "layer", "entry": "forward", "T": 1, "bias": 0.0},
        # the MoE of one decoded token through the whole model
        {"name": "decode_1_stack40", "kind": "stack", "layers": 40, "T": 1},
        # a decode step that verifies three drafted tokens with the last one
        {"name": "decode_4_stack40", "kind": "stack", "layers": 40, "T": 4},
        # eight sequences decoded together, skewed routing
        {"name": "decode_8_layer", "kind": "layer", "entry": "normed", "T": 8, "bias": 1.0},
        # a dozen sequences, or a short question's first chunk
        {"name": "prefill_12_layer", "kind": "layer", "entry": "forward", "T": 12, "bias": 0.0},
        # a chat turn
        {"name": "prefill_100_layer", "kind": "layer", "entry": "forward", "T": 100, "bias": 0.0},
        # the benchmark's 512-token prompt
        {"name": "prefill_512_layer", "kind": "layer", "entry": "normed", "T": 512, "bias": 1.0},
        # a ragged prompt with the next block's norm fused in
        {"name": "prefill_1999_layer", "kind": "layer", "entry": "norm", "T": 1999, "bias": 0.0},
        # the benchmark's long prompt, heavily skewed routing
        {"name": "prefill_8192_layer", "kind": "layer", "entry": "normed", "T": 8192, "bias": 1.3},
        # one bf16 matrix of one expert: the converter on a small tensor
        {"name": "rows_bf16", "kind": "rows", "src": "bf16", "rows": 512, "cols": 2048},
        # the converter on a layer of experts, from the Q8_0 files it usually gets
        {"name": "convert_q8_0", "kind": "convert", "src": "q8_0"},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    r = rng.random()
    if r < 0.65:
        return {"kind": "layer", "entry": rng.choice(("normed", "forward", "norm")), "T": spread(1, 8191),
                "bias": rng.choice((0.0, 0.7, 1.0, 1.3))}
    if r < 0.85:
        return {"kind": "stack", "layers": rng.randint(2, 39), "T": rng.randint(1, 8)}
    return {"kind": "rows", "src": rng.choice(sorted(SOURCES)), "rows": spread(3, 130000),
            "cols": 256 * rng.choice((1, 2, 3, 5, 8))}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _half_bytes(t):
    return t.half().view(torch.uint8)


def _layer_weights(g, bias):
    """One layer's tensors on the GPU, in the formats the library takes."""
    def normal(*shape):
        return torch.randn(shape, device="cuda", generator=g)

    blobs = torch.randint(0, 256, (E, EXPERT), dtype=torch.uint8, device="cuda", generator=g)
    gu = blobs[:, :DOWN].view(E, 2 * FF, GU_ROW)
    dn = blobs[:, DOWN:].view(E, D, DN_ROW)
    # codes are uniform, so codebook values have an rms of 70
    for rows, cols in ((gu, D), (dn, FF)):
        n = rows.shape[1]
        scale = (0.5 + torch.rand((E, n, cols // BLK), device="cuda", generator=g)) * (0.02 / 70)
        rows[:, :, cols // 2:] = _half_bytes(scale)

    def q8(rows, cols):
        w = torch.empty((rows, cols + cols // BLK * 2), dtype=torch.uint8, device="cuda")
        w[:, :cols] = torch.randint(-127, 128, (rows, cols), device="cuda", generator=g).to(torch.int8).view(torch.uint8)
        scale = (0.5 + torch.rand((rows, cols // BLK), device="cuda", generator=g)) * (0.02 / 73)
        w[:, cols:] = _half_bytes(scale)
        return w

    w = {"blobs": blobs, "post_norm": 1.0 + 0.1 * normal(D), "router": 0.02 * normal(257, D), "sh_gu": q8(1024, D),
         "sh_down": q8(D, FF), "bias": None}
    if bias:
        rank = torch.randperm(E, device="cuda", generator=g).double() + 1.0
        w["bias"] = (-bias * rank.log()).float()
    return w


def _set_layer(m, layer, w, st):
    m.upload_experts(layer, 0, w["blobs"], on_device=True, stream=st)
    m.set_dense(layer, post_norm=w["post_norm"], router=w["router"], bias=w["bias"], sh_gu=w["sh_gu"],
                sh_down=w["sh_down"], on_device=True, stream=st)


def _activations(case, g):
    x = torch.randn((case["T"], D), device="cuda", generator=g)
    nw = 1.0 + 0.1 * torch.randn(D, device="cuda", generator=g) if case.get("entry") == "norm" else None
    return x, nw


def _source(src, nblk, g):
    """nblk 32-blocks of weights of rms about 0.02, as ggml stores them in type `src`."""
    if src == "q8_0":
        b = torch.randint(0, 256, (nblk, 34), dtype=torch.uint8, device="cuda", generator=g)
        b[:, :2] = _half_bytes((0.5 + torch.rand((nblk, 1), device="cuda", generator=g)) * (0.02 / 73))
        return b
    w = 0.02 * torch.randn(nblk * BLK, device="cuda", generator=g)
    return w.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[src])


class _Device:
    """A torch view of memory the library owns."""

    def __init__(self, ptr, nbytes, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 3}


def prepare(case, seed):
    g = _generator(seed)
    st = torch.cuda.current_stream()
    if case["kind"] in ("layer", "stack"):
        n = case.get("layers", 1)
        m = qe_moe.MoE(n_layers=n, t_max=case["T"])
        x, nw = _activations(case, g)
        for layer in range(n):
            _set_layer(m, layer, _layer_weights(g, case.get("bias", 0.0)), st)
        return {"case": case, "m": m, "x": x, "nw": nw, "y": torch.empty_like(x),
                "xn": torch.empty_like(x) if nw is not None else None}
    if case["kind"] == "rows":
        cols = case["cols"]
        return {"case": case, "src": _source(case["src"], case["rows"] * cols // BLK, g),
                "dst": torch.empty((case["rows"], cols // 2 + cols // BLK * 2), dtype=torch.uint8, device="cuda")}
    m = qe_moe.MoE(n_layers=1, t_max=1)
    n = E * FF * D // BLK
    return {"case": case, "m": m, "gate": _source(case["src"], n, g), "up": _source(case["src"], n, g),
            "down": _source(case["src"], n, g),
            "arena": torch.as_tensor(_Device(m.arena_ptr(0), E * EXPERT, m), device="cuda")}


def run(s):
    case = s["case"]
    st = torch.cuda.current_stream()
    if case["kind"] == "rows":
        qe_moe.nl4_quantize_rows(s["src"], SOURCES[case["src"]][0], case["rows"], case["cols"], s["dst"], stream=st)
        return s["dst"]
    m = s["m"]
    if case["kind"] == "convert":
        m.convert_experts(0, s["gate"], s["up"], s["down"], SOURCES[case["src"]][0], stream=st)
        return s["arena"]
    if case["kind"] == "stack":
        m.forward_stack(0, case["layers"], s["x"], s["y"], case["T"], stream=st)
        return s["y"]
    if case["entry"] == "normed":
        m.forward_normed(0, s["x"], s["y"], case["T"], stream=st)
        return s["y"]
    if case["entry"] == "forward":
        m.forward(0, s["x"], s["y"], case["T"], stream=st)
        return s["y"]
    m.forward_norm(0, s["x"], s["y"], case["T"], s["nw"], s["xn"], stream=st)
    return {"y": s["y"], "xn": s["xn"]}


def _distinct_experts(T, bias):
    """Experts that T tokens reach, from random logits of the router's spread (0.02 * sqrt(2048))."""
    r = np.random.default_rng(7)
    logits = r.standard_normal((T, E), dtype=np.float32) * np.float32(0.905)
    logits -= np.float32(bias) * np.log(np.arange(1, E + 1, dtype=np.float32))
    return int(np.unique(np.argpartition(logits, E - K, axis=1)[:, E - K:]).size)


def work(case):
    if case["kind"] == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": n // BLK * (SOURCES[case["src"]][1] + 18), "flops": n * 16 * 4}  # 16 candidate scales, 2 sums
    if case["kind"] == "convert":
        n = 3 * E * FF * D
        return {"bytes": n // BLK * (SOURCES[case["src"]][1] + 18), "flops": n * 16 * 4}
    T, n = case["T"], case.get("layers", 1)
    rows = {"normed": 2, "forward": 2, "norm": 3}[case.get("entry", "forward")]
    return {"bytes": n * (_distinct_experts(T, case.get("bias", 0.0)) * EXPERT + DENSE) + rows * T * D * 4,
            "flops": n * T * FLOP_TOKEN}


def tolerance(case):
    if case["kind"] in ("rows", "convert"):
        return "exact"
    # Measured against exact(): up to 1.3e-4 for a layer and 4.7e-3 for a stack, all
    # of it int8 activations that land on the other side of a rounding step (and,
    # through many layers, a token's eighth expert with them).  Four times that is
    # what another order of the fp32 sums could show.
    return {"rel": 0.015} if case["kind"] == "stack" else {"rel": 5e-4}


def _nl4(rows, cols):
    """IQ4_NL rows (uint8) as float64."""
    codes = rows[:, : cols // 2].reshape(-1, cols // BLK, 16)
    scale = rows[:, cols // 2:].contiguous().view(torch.float16).double()
    book = torch.tensor(CODEBOOK, dtype=torch.float64, device=rows.device)
    w = torch.cat((book[(codes & 15).long()], book[(codes >> 4).long()]), dim=2)
    return (w * scale[:, :, None]).reshape(-1, cols)


def _q8(rows, cols):
    scale = rows[:, cols:].contiguous().view(torch.float16).double()
    q = rows[:, :cols].contiguous().view(torch.int8).double().view(-1, cols // BLK, BLK)
    return (q * scale[:, :, None]).reshape(-1, cols)


def _int8(x):
    """x as the library's int8 activations hold it: per 32-block, a scale of amax / 127."""
    b = x.reshape(x.shape[0], -1, BLK)
    d = b.abs().amax(dim=2, keepdim=True) / 127.0
    q = torch.where(d > 0, torch.round(b / torch.where(d > 0, d, 1.0)), 0.0)
    return (q * d).reshape(x.shape)


def _silu(g):
    return g / (1.0 + torch.exp(-g))


def _rmsnorm(x, w):
    return x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS) * w.double()


def _moe64(w, xn):
    logits = xn @ w["router"].double().t().contiguous()
    routed = logits[:, :E]
    if w["bias"] is not None:
        routed = routed + w["bias"].double()
    top, ids = routed.topk(K, dim=1)
    wts = torch.softmax(top, dim=1)
    gu = _q8(w["sh_gu"], D)
    h = _silu(xn @ gu[:FF].t().contiguous()) * (xn @ gu[FF:].t().contiguous())
    y = torch.sigmoid(logits[:, E:]) * (h @ _q8(w["sh_down"], FF).t().contiguous())
    xq = _int8(xn)
    for e in ids.unique().tolist():
        tok, k = (ids == e).nonzero(as_tuple=True)
        rows = _nl4(w["blobs"][e, :DOWN].view(2 * FF, GU_ROW), D)
        gu = xq[tok] @ rows.t().contiguous()
        h = _int8(_silu(gu[:, :FF]) * gu[:, FF:])
        down = _nl4(w["blobs"][e, DOWN:].view(D, DN_ROW), FF)
        y.index_add_(0, tok, (h @ down.t().contiguous()) * wts[tok, k][:, None])
    return y


def exact(case, seed):
    if case["kind"] in ("rows", "convert"):
        return None
    g = _generator(seed)
    x, nw = _activations(case, g)
    y = x.double()
    for _ in range(case.get("layers", 1)):
        w = _layer_weights(g, case.get("bias", 0.0))
        if case.get("entry") == "normed":
            y = _moe64(w, y)
        else:
            y = y + _moe64(w, _rmsnorm(y, w["post_norm"]))
    return {"y": y, "xn": _rmsnorm(y, nw)} if nw is not None else y
