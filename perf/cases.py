"""The work that an SDXL program has this library do, as measurable cases.

A case is a dict of plain values; `prepare` makes its inputs on the GPU,
`run` is one pass through the package's entry points (sdvk_amd.ops), `work`
the bytes and operations the pass cannot do without, `exact` the same result
in 64 bits, `tolerance` how far another correct implementation may be from it.

Buffers are torch tensors handed over by address, so the library is bound to
the HIP runtime that torch has loaded: one runtime, one default stream.

Image sizes run from 512 to 1536 pixels a side in steps of 64, up to a megapixel; a UNet level of
640 channels then has (H / 16) x (W / 16) tokens and one of 1280 channels
(H / 32) x (W / 32), times one or two guidance rows. The context is 77 tokens
a prompt chunk of 2048 channels.
"""
from __future__ import annotations

import math
from pathlib import Path

import torch

from sdvk_amd import hip, ops

# The HIP runtime of this process is torch's: a second one (the package's
# default, ROCm's own) would not know torch's buffers or streams.
hip.ROCM = Path(torch.__file__).resolve().parent

DEV = "cuda"
CTX_TOKENS, CTX_CHANNELS = 77, 2048
LINEARS = [(640, 640), (1280, 1280), (640, 2560), (1280, 5120)]      # (N, K): q / k / v / out, FF-down
CONVS = [(320, 2880), (640, 2880), (640, 5760), (1280, 5760), (1280, 11520), (640, 320), (1280, 640)]  # (M, K)
BLOCK_FLAGS = (ops.MI_BLOCK_FUSED_EPILOGUES | ops.MI_BLOCK_JOINT_QKV | ops.MI_BLOCK_FP16_ACTIVATIONS |
               ops.MI_BLOCK_FP16_ATTENTION)


def listed():
    return [
        # a ResBlock's time-embedding projection, two guidance rows: the smallest linear of a step
        dict(name="temb_2x1280x1280", kind="linear", M=2, N=1280, K=1280, layout="split", act="f32", bias=True, ws=True),
        # cross-attention K or V of two 77-token prompts, 34-byte blocks, K split over a workspace
        dict(name="xkv_154x1280x2048", kind="linear", M=154, N=1280, K=2048, layout="blocks", act="f32", bias=False, ws=True),
        # an attention projection at 768 x 768 (2 x 24 x 24 tokens), fp32 activations
        dict(name="proj_1152x1280x1280", kind="linear", M=1152, N=1280, K=1280, layout="blocks", act="f32", bias=True, ws=True),
        # the reference's GEMM benchmark shape in its own weight layout
        dict(name="split_9216x1280x1280", kind="linear", M=9216, N=1280, K=1280, layout="split", act="f32", bias=False, ws=False),
        # FF-down at 1024 x 1024 from fp16 activations
        dict(name="ffdown_2048x1280x5120", kind="linear", M=2048, N=1280, K=5120, layout="blocks", act="f16", bias=True, ws=True),
        # FF-up with GEGLU at 832 x 1216 (2 x 26 x 38 tokens), fp16 activations in and out
        dict(name="geglu_1976x5120x1280", kind="geglu", M=1976, F=5120, K=1280, act="f16"),
        # a 3 x 3 convolution of 640 channels at 1024 x 1024 after im2col (64 x 64 pixels)
        dict(name="conv_640x4096x5760", kind="conv", M=640, N=4096, K=5760),
        # self-attention of the 640-channel level at 1024 x 1024, fp16, both guidance rows
        dict(name="self_f16_2x10x4096", kind="attn", entry="ws", batch=2, heads=10, Tq=4096, Tk=4096, causal=False, masked=False),
        # cross-attention of the 1280-channel level, fp16, prompts padded to 77 tokens
        dict(name="cross_f16_2x20x1024x77", kind="attn", entry="ws", batch=2, heads=20, Tq=1024, Tk=77, causal=False, masked=True),
        # the reference's attention call (fp32, one guidance row) at 768 x 768
        dict(name="self_f32_10x2304", kind="attn", entry="fused", batch=1, heads=10, Tq=2304, Tk=2304, causal=False, masked=False),
        # one transformer block of the 1280-channel level at 832 x 1216 as a sampler runs it: every fast option, K / V cached
        dict(name="block_fast_2x988x1280", kind="block", batch=2, tokens=988, C=1280, fast=True),
        # one transformer block of the 640-channel level at 1024 x 1024 in the reference's sequence of operators
        dict(name="block_plain_2x4096x640", kind="block", batch=2, tokens=4096, C=640, fast=False),
    ]


def draw(rng):
    h, w = 64 * rng.randint(8, 24), 64 * rng.randint(8, 24)
    while h * w > 1024 * 1024:  # trained sizes: a megapixel at most
        h, w = 64 * rng.randint(8, 24), 64 * rng.randint(8, 24)
    rows = rng.choice([1, 2, 2])
    C = rng.choice([640, 1280])
    tokens = (h // 16) * (w // 16) if C == 640 else (h // 32) * (w // 32)
    kind = rng.choice(["temb", "xkv", "linear", "linear", "split", "geglu", "conv", "self", "cross", "fused", "block", "plain"])
    if kind == "temb":
        N, K = rng.choice([(320, 1280), (640, 1280), (1280, 1280), (1280, 320), (1280, 2816)])
        return dict(kind="linear", M=rng.randint(1, 8), N=N, K=K, layout=rng.choice(["split", "blocks"]), act="f32",
                    bias=True, ws=rng.random() < 0.5)
    if kind == "xkv":
        return dict(kind="linear", M=CTX_TOKENS * rng.randint(1, 4), N=C, K=CTX_CHANNELS, layout="blocks", act="f32",
                    bias=False, ws=True)
    if kind == "linear":
        N, K = rng.choice([s for s in LINEARS if s[0] == C])
        return dict(kind="linear", M=rows * tokens, N=N, K=K, layout="blocks", act=rng.choice(["f32", "f16"]),
                    bias=rng.random() < 0.7, ws=True)
    if kind == "split":
        N, K = rng.choice([(C, C), (8 * C, C), (C, 4 * C)])
        return dict(kind="linear", M=rows * tokens, N=N, K=K, layout="split", act="f32", bias=rng.random() < 0.5,
                    ws=rng.random() < 0.5)
    if kind == "geglu":
        return dict(kind="geglu", M=rows * tokens, F=4 * C, K=C, act=rng.choice(["f32", "f16"]))
    if kind == "conv":
        M, K = rng.choice(CONVS)
        side = 8 if M == 320 else 16 if M == 640 else 32
        return dict(kind="conv", M=M, N=max(4, min(4096, (h // side) * (w // side)) // 4 * 4), K=K)
    if kind == "self":
        return dict(kind="attn", entry="ws", batch=rows, heads=C // 64, Tq=tokens, Tk=tokens, causal=False, masked=False)
    if kind == "cross":
        return dict(kind="attn", entry="ws", batch=rows, heads=C // 64, Tq=tokens, Tk=CTX_TOKENS * rng.randint(1, 3),
                    causal=False, masked=rng.random() < 0.7)
    if kind == "fused":
        if rng.random() < 0.3:  # a text encoder's causal self-attention
            return dict(kind="attn", entry="fused", batch=1, heads=rng.choice([12, 20]), Tq=CTX_TOKENS, Tk=CTX_TOKENS,
                        causal=True, masked=False)
        return dict(kind="attn", entry="fused", batch=1, heads=C // 64, Tq=tokens,
                    Tk=rng.choice([tokens, tokens, CTX_TOKENS]), causal=False, masked=False)
    return dict(kind="block", batch=rows, tokens=tokens, C=C, fast=kind == "block")


# ------------------------------------------------------------------ inputs --

class Buf:
    """A device buffer as the entry points take one: its address and its size in bytes."""

    def __init__(self, nbytes):
        self.t = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=DEV)
        self.value, self.nbytes = self.t.data_ptr(), int(nbytes)


def normal(g, *shape, std=1.0):
    x = torch.empty(*shape, device=DEV).normal_(generator=g)
    return x.mul_(std) if std != 1.0 else x


def quantize(w):
    """(d fp16 [blocks, 1], q int8 [blocks, 32]) of an fp32 weight, the GGUF rule."""
    b = w.reshape(-1, 32)
    amax = b.abs().amax(1, keepdim=True)
    q = torch.round(b * torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))).clamp(-127, 127).to(torch.int8)
    return (amax / 127.0).to(torch.float16), q


def blocks_of(w):
    """The 34-byte GGUF Q8_0 blocks of an fp32 weight, as bytes."""
    d, q = quantize(w)
    return torch.cat([d.view(torch.uint8).reshape(-1, 2), q.view(torch.uint8)], 1).reshape(-1)


def value64(raw):
    """float64 values of 34-byte blocks."""
    b = raw.reshape(-1, 34)
    d = b[:, :2].contiguous().view(torch.float16).double()
    return (b[:, 2:].contiguous().view(torch.int8).double() * d).reshape(-1)


def generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def linear_inputs(c, seed):
    g = generator(seed)
    M, N, K = c["M"], c["N"], c["K"]
    x = normal(g, M, K)
    w = normal(g, N, K, std=0.02)
    s = dict(A=x.half() if c["act"] == "f16" else x, bias=normal(g, N, std=0.02) if c["bias"] else None)
    if c["layout"] == "split":
        d, q = quantize(w)
        s["q"], s["d"] = q.reshape(-1), d.float().reshape(-1)
    else:
        s["W"] = blocks_of(w)
    return s


def geglu_inputs(c, seed):
    g = generator(seed)
    x = normal(g, c["M"], c["K"])
    return dict(A=x.half() if c["act"] == "f16" else x, W=blocks_of(normal(g, 2 * c["F"], c["K"], std=0.02)),
                bias=normal(g, 2 * c["F"], std=0.02))


def conv_inputs(c, seed):
    g = generator(seed)
    d, q = quantize(normal(g, c["M"], c["K"], std=0.02))
    return dict(q=q.reshape(-1), d=d.float().reshape(-1), B=normal(g, c["K"], c["N"]))


def attn_inputs(c, seed):
    g = generator(seed)
    C, dt = 64 * c["heads"], torch.float32 if c["entry"] == "fused" else torch.float16
    q, k, v = (normal(g, c["batch"], t, C).to(dt) for t in (c["Tq"], c["Tk"], c["Tk"]))
    lens = torch.randint(1, c["Tk"] + 1, (c["batch"],), generator=g, device=DEV, dtype=torch.int32) if c["masked"] else None
    return dict(q=q, k=k, v=v, lens=lens)


MATS = {"attn1_q": 1, "attn1_k": 1, "attn1_v": 1, "attn1_out": 1, "attn2_q": 1, "attn2_k": 0, "attn2_v": 0, "attn2_out": 1}


def block_inputs(c, seed):
    g = generator(seed)
    C, F = c["C"], 4 * c["C"]
    s = dict(x=normal(g, c["batch"] * c["tokens"], C), ctx=normal(g, c["batch"] * CTX_TOKENS, CTX_CHANNELS))
    shapes = {n: (C, C if own else CTX_CHANNELS) for n, own in MATS.items()} | {"ff_up": (2 * F, C), "ff_down": (C, F)}
    w = {n: blocks_of(normal(g, *shape, std=0.02)) for n, shape in shapes.items()}
    w["qkv"] = torch.cat([w.pop("attn1_q"), w.pop("attn1_k"), w.pop("attn1_v")])  # one [3C, C] matrix
    for n, size in (("attn1_out_b", C), ("attn2_out_b", C), ("ff_up_b", 2 * F), ("ff_down_b", C)):
        w[n] = normal(g, size, std=0.02)
    for i in (1, 2, 3):
        w[f"norm{i}_w"], w[f"norm{i}_b"] = 1 + normal(g, C, std=0.1), normal(g, C, std=0.1)
    s["w"] = w
    return s


INPUTS = {"linear": linear_inputs, "geglu": geglu_inputs, "conv": conv_inputs, "attn": attn_inputs, "block": block_inputs}


def prepare(case, seed):
    c = case
    s = INPUTS[c["kind"]](c, seed)
    s["case"], s["kind"] = c, c["kind"]
    if c["kind"] == "linear":
        s["C"] = torch.empty(c["M"], c["N"], device=DEV)
        n = ops.gemm_workspace_bytes(c["M"], c["N"], c["K"]) if c["ws"] else 0
        s["ws"] = Buf(n) if n else None
    elif c["kind"] == "geglu":
        s["G"] = torch.empty(c["M"], c["F"], device=DEV, dtype=s["A"].dtype)
    elif c["kind"] == "conv":
        s["C"] = torch.empty(c["M"], c["N"], device=DEV)
        n = ops.gemm_nn_workspace_bytes(c["M"], c["N"], c["K"])
        s["ws"] = Buf(n) if n else None
    elif c["kind"] == "attn":
        s["o"] = torch.empty_like(s["q"])
        if c["entry"] == "ws":
            s["args"] = dict(batch=c["batch"], Tq=c["Tq"], Tk=c["Tk"], C=64 * c["heads"], heads=c["heads"],
                             causal=c["causal"], in_dtype=ops.MI_F16, out_dtype=ops.MI_F16,
                             kv_len=s["lens"].data_ptr() if s["lens"] is not None else None)
            n = ops.fused_attention_ws_bytes(**s["args"])
            s["ws"] = Buf(n) if n else None
        else:
            s["args"] = ops.FusedAttnArgs(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr(),
                                          c["Tq"], c["Tk"], 64 * c["heads"], c["heads"], c["causal"])
    else:
        C, w = c["C"], s["w"]
        p = {n: t.data_ptr() for n, t in w.items() if n != "qkv"}
        for i, n in enumerate(("attn1_q", "attn1_k", "attn1_v")):
            p[n] = w["qkv"].data_ptr() + i * (C * (C // 32) * 34)
        s["weights"] = ops.BlockWeights(**p)
        s["dims"] = ops.BlockDims(c["batch"], c["tokens"], C, C // 64, CTX_TOKENS, CTX_CHANNELS, 4 * C,
                                  BLOCK_FLAGS if c["fast"] else 0)
        s["ws"] = Buf(ops.block_workspace_bytes(s["dims"]))
        s["t"] = torch.empty_like(s["x"])  # the residual stream the block updates in place
        if c["fast"]:
            # the context is fixed for a sampling job: its K / V are made once, before the steps
            s["kv"] = Buf(ops.block_ctx_kv_bytes(s["dims"]))
            ops.block_ctx_kv(s["weights"], s["dims"], s["ctx"].data_ptr(), s["kv"])
    return s


# -------------------------------------------------------------------- pass --

def address(t):
    return t.data_ptr() if t is not None else None


def run(state):
    s = state
    c = s["case"]
    if s["kind"] == "linear":
        a = (c["M"], c["N"], c["K"])
        if c["layout"] == "split":
            if c["bias"]:
                ops.gemm_nt_q8_bias(s["A"].data_ptr(), s["q"].data_ptr(), s["C"].data_ptr(), s["d"].data_ptr(),
                                    s["bias"].data_ptr(), *a, workspace=s["ws"])
            else:
                ops.gemm_nt_q8(s["A"].data_ptr(), s["q"].data_ptr(), s["C"].data_ptr(), s["d"].data_ptr(), *a,
                               workspace=s["ws"])
        else:
            gemm = ops.gemm_nt_q8_0_f16a if c["act"] == "f16" else ops.gemm_nt_q8_0
            gemm(s["A"].data_ptr(), s["W"].data_ptr(), s["C"].data_ptr(), *a, bias=address(s["bias"]), workspace=s["ws"])
        return s["C"]
    if s["kind"] == "geglu":
        f = ops.gemm_nt_q8_0_geglu_f16 if c["act"] == "f16" else ops.gemm_nt_q8_0_geglu
        f(s["A"].data_ptr(), s["W"].data_ptr(), s["G"].data_ptr(), c["M"], c["F"], c["K"], bias=s["bias"].data_ptr())
        return s["G"]
    if s["kind"] == "conv":
        ops.gemm_nn_q8(s["q"].data_ptr(), s["d"].data_ptr(), s["B"].data_ptr(), s["C"].data_ptr(), c["M"], c["N"],
                       c["K"], workspace=s["ws"])
        return s["C"]
    if s["kind"] == "attn":
        if c["entry"] == "ws":
            ops.fused_attention_ws(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr(), s["ws"],
                                   **s["args"])
        else:
            ops.fused_attention(s["args"])
        return s["o"]
    s["t"].copy_(s["x"])  # a step's hidden state arrives; the block updates it in place
    if c["fast"]:
        ops.sdxl_block_forward_kv(s["weights"], s["dims"], s["t"].data_ptr(), s["kv"], s["ws"])
    else:
        ops.sdxl_block_forward(s["weights"], s["dims"], s["t"].data_ptr(), s["ctx"].data_ptr(), s["ws"])
    return s["t"]


# ---------------------------------------------------------- floor and bars --

def work(case):
    c = case
    if c["kind"] == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        wb = N * K * (1 + 4 / 32 if c["layout"] == "split" else 34 / 32)
        return {"bytes": M * K * (2 if c["act"] == "f16" else 4) + wb + 4 * M * N + (4 * N if c["bias"] else 0),
                "flops": 2.0 * M * N * K}
    if c["kind"] == "geglu":
        M, F, K, e = c["M"], c["F"], c["K"], 2 if c["act"] == "f16" else 4
        return {"bytes": M * K * e + 2 * F * K * 34 / 32 + 8 * F + M * F * e, "flops": 4.0 * M * F * K}
    if c["kind"] == "conv":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": M * K * (1 + 4 / 32) + 4.0 * K * N + 4.0 * M * N, "flops": 2.0 * M * N * K}
    if c["kind"] == "attn":
        C, e = 64 * c["heads"], 4 if c["entry"] == "fused" else 2
        return {"bytes": e * c["batch"] * C * 2.0 * (c["Tq"] + c["Tk"]),
                "flops": 4.0 * c["batch"] * c["Tq"] * c["Tk"] * C * (0.5 if c["causal"] else 1.0)}
    B, T, C = c["batch"], c["tokens"], c["C"]
    rows, ctx = B * T, B * CTX_TOKENS
    linear = 2.0 * rows * C * (6 * C + 12 * C) + (0.0 if c["fast"] else 4.0 * ctx * CTX_CHANNELS * C)
    weights = (6 + 12) * C * C + (0 if c["fast"] else 2 * CTX_CHANNELS * C)
    return {"bytes": 8.0 * rows * C + weights * 34 / 32 + (4 * ctx * C if c["fast"] else 4 * ctx * CTX_CHANNELS),
            "flops": linear + 4.0 * B * T * (T + CTX_TOKENS) * C}


def tolerance(case):
    c = case
    if c["kind"] == "attn":
        # fp32 in and out: split into fp16 parts, 32-bit sums; fp16: the output's own rounding and the weights'
        return {"rel": 4e-6} if c["entry"] == "fused" else {"rel": 1.2e-3}
    if c["kind"] == "block":
        # the residual stream passes the block unrounded, so its relative error is under its operators'
        return {"rel": 9e-4}
    # operands rounded to fp16, 32-bit sums; GEGLU multiplies two such results
    return {"rel": 1.5e-3 if c["kind"] == "geglu" else 1.2e-3}


# ------------------------------------------------------------ 64-bit result --

def matmul64(a, raw, N, K):
    return a.double() @ value64(raw).reshape(N, K).t().contiguous()


def attention64(q, k, v, heads, lens=None, causal=False):
    """[B, T, C] attention in 64 bits, one head of one row at a time."""
    B, Tq, C = q.shape
    Tk, d = k.shape[1], C // heads
    o = torch.zeros(B, Tq, C, dtype=torch.float64, device=q.device)
    for b in range(B):
        L = Tk if lens is None else int(lens[b])
        for h in range(heads):
            cols = slice(h * d, (h + 1) * d)
            kt = k[b, :L, cols].double().t().contiguous()
            sc = (q[b, :, cols].double() @ kt) / math.sqrt(d)
            if causal:
                sc.masked_fill_(torch.ones(Tq, L, dtype=torch.bool, device=q.device).triu(1), -math.inf)
            o[b, :, cols] = torch.softmax(sc, -1) @ v[b, :L, cols].double().contiguous()
    return o


def norm64(x, w, b):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w.double(), b.double(), 1e-5)


def gelu64(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2.0)))


def exact(case, seed):
    c = case
    s = INPUTS[c["kind"]](c, seed)
    if c["kind"] == "linear":
        if c["layout"] == "split":
            w = (s["q"].double().reshape(-1, 32) * s["d"].double().reshape(-1, 1)).reshape(c["N"], c["K"])
            y = s["A"].double() @ w.t().contiguous()
        else:
            y = matmul64(s["A"], s["W"], c["N"], c["K"])
        return y if s["bias"] is None else y + s["bias"].double()
    if c["kind"] == "geglu":
        y = matmul64(s["A"], s["W"], 2 * c["F"], c["K"]) + s["bias"].double()
        return y[:, :c["F"]] * gelu64(y[:, c["F"]:])
    if c["kind"] == "conv":
        w = (s["q"].double().reshape(-1, 32) * s["d"].double().reshape(-1, 1)).reshape(c["M"], c["K"])
        return w @ s["B"].double()
    if c["kind"] == "attn":
        return attention64(s["q"], s["k"], s["v"], c["heads"], s["lens"], c["causal"])
    B, T, C, w = c["batch"], c["tokens"], c["C"], s["w"]
    H, x, n1 = C // 64, s["x"].double(), C * (C // 32) * 34
    q, k, v = (w["qkv"][i * n1:(i + 1) * n1] for i in range(3))

    def rows(y, t):
        return y.reshape(B, t, C)

    n = norm64(x, w["norm1_w"], w["norm1_b"])
    o = attention64(*(rows(matmul64(n, m, C, C), T) for m in (q, k, v)), H)
    x = x + matmul64(o.reshape(-1, C), w["attn1_out"], C, C) + w["attn1_out_b"].double()
    n = norm64(x, w["norm2_w"], w["norm2_b"])
    o = attention64(rows(matmul64(n, w["attn2_q"], C, C), T),
                    *(rows(matmul64(s["ctx"], w[m], C, CTX_CHANNELS), CTX_TOKENS) for m in ("attn2_k", "attn2_v")), H)
    x = x + matmul64(o.reshape(-1, C), w["attn2_out"], C, C) + w["attn2_out_b"].double()
    n = norm64(x, w["norm3_w"], w["norm3_b"])
    y = matmul64(n, w["ff_up"], 8 * C, C) + w["ff_up_b"].double()
    g = y[:, :4 * C] * gelu64(y[:, 4 * C:])
    return x + matmul64(g, w["ff_down"], C, 4 * C) + w["ff_down_b"].double()
