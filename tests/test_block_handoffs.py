"""The block's fused epilogues and fp16 hand-offs against separate fp32 operators,
bit for bit, by alignment: an x or a LayerNorm parameter that is not 16-byte
aligned takes fp32 hand-offs (an error only where MI_BLOCK_FP16_ACTIVATIONS asks
for fp16). Head dims that are no multiple of 8 take the element-wise attention."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_block import make_weights, to_device

pytestmark = pytest.mark.gpu


def separate(w, x, ctx, B, T, C, H, Tc, Cc, F):
    """The block's operators one entry each on pointers w / x, every hand-off fp32; x in place."""
    from sdvk_amd import ops
    from sdvk_amd.hip import DeviceBuffer

    R = B * T
    buf = {k: DeviceBuffer(4 * n) for k, n in dict(n=R * C, q=R * C, k=max(R, B * Tc) * C, v=max(R, B * Tc) * C,
                                                   o=R * C, a=R * C, h=2 * R * F, g=R * F).items()}
    split = [DeviceBuffer(max(16, ops.gemm_workspace_bytes(R, C, K))) for K in (C, F)]

    def attn(tk):
        ops.fused_attention_ex(buf["q"], buf["k"], buf["v"], buf["o"], batch=B, Tq=T, Tk=tk, C=C, heads=H,
                               precision=ops.MI_ATTN_PREC_FP16)

    def residual(a, name, K):
        ops.gemm_nt_q8_0(buf[a], w[name], buf["a"], R, C, K, bias=w[name + "_b"], workspace=split[K == F])
        ops.add2(x, buf["a"], R * C)

    def norm(i):
        ops.layernorm(x, w[f"norm{i}_w"], w[f"norm{i}_b"], buf["n"], R, C)

    norm(1)
    for n in "qkv":
        ops.gemm_nt_q8_0(buf["n"], w["attn1_" + n], buf[n], R, C, C)
    attn(T)
    residual("o", "attn1_out", C)
    norm(2)
    ops.gemm_nt_q8_0(buf["n"], w["attn2_q"], buf["q"], R, C, C)
    for n in "kv":
        ops.gemm_nt_q8_0(ctx, w["attn2_" + n], buf[n], B * Tc, C, Cc)
    attn(Tc)
    residual("o", "attn2_out", C)
    norm(3)
    ops.gemm_nt_q8_0(buf["n"], w["ff_up"], buf["h"], R, 2 * F, C, bias=w["ff_up_b"])
    ops.geglu(buf["h"], buf["g"], R, F)
    residual("g", "ff_down", F)


@pytest.mark.parametrize("B,T,C,H,Tc,Cc,F", [(2, 40, 128, 2, 77, 256, 256), (1, 33, 96, 8, 5, 96, 160),
                                             (1, 9, 64, 1, 5, 96, 160)])
@pytest.mark.parametrize("moved", [None, "x", "norm2_b"])
def test_handoffs(gpu, oracle, B, T, C, H, Tc, Cc, F, moved):
    from sdvk_amd import ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    w = make_weights(oracle, C, Cc, F, seed=700)
    dev, _ = to_device(w)
    x, ctx = oracle.normal(1, B * T * C), DeviceBuffer.from_array(oracle.normal(2, B * Tc * Cc))
    pad = lambda a: DeviceBuffer.from_array(np.concatenate([np.zeros(1, np.float32), a]))
    keep = pad(w["norm2_b"])
    ptrs = {k: b.value for k, b in dev.items()}
    if moved == "norm2_b":
        ptrs[moved] = keep.value + 4
    off = 1 if moved == "x" else 0

    def run(f):
        dx = pad(x) if off else DeviceBuffer.from_array(x)
        f(dx.value + 4 * off)
        synchronize()
        return dx.download(np.float32, x.size, offset=4 * off)

    def block(flags):
        dims = ops.BlockDims(B, T, C, H, Tc, Cc, F, flags)
        ws = DeviceBuffer(ops.block_workspace_bytes(dims))
        def f(xp):
            ops.sdxl_block_forward(ops.BlockWeights(**ptrs), dims, xp, ctx, ws)
            synchronize()
        return f

    ref = run(lambda xp: separate(ptrs, xp, ctx, B, T, C, H, Tc, Cc, F))
    assert np.all(np.isfinite(ref)) and not np.array_equal(ref, x)
    assert np.array_equal(run(block(0)), ref)
    half = block(ops.MI_BLOCK_FP16_ACTIVATIONS | ops.MI_BLOCK_FUSED_EPILOGUES)
    if moved:
        with pytest.raises(ops.MiError):
            run(half)
    else:
        assert np.array_equal(run(half), ref)
