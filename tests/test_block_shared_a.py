"""Several weights on one A in one launch (a block's Q / K / V, its context K / V)
against the GEMM entry one weight at a time, bit for bit: few rows, tiles of
every size, fp16 context K / V. On the CPU the block cases of the kernel
emulator cover the same launches with guard pages."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import q8_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Tc,C,Cc", [(1, 5, 64, 96), (2, 77, 640, 2048), (2, 77, 320, 1024), (4, 77, 1280, 2048)])
@pytest.mark.parametrize("half", [False, True])
def test_context_kv(gpu, oracle, B, Tc, C, Cc, half):
    from sdvk_amd import ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    w = {n: DeviceBuffer.from_array(q8_weights(oracle, i, C, Cc)) for i, n in enumerate(("attn2_k", "attn2_v"))}
    any_w = w["attn2_k"]
    bw = ops.BlockWeights(**{f: w.get(f, any_w) for f in ops.BlockWeights.__dataclass_fields__})
    dims = ops.BlockDims(B, 64, C, max(1, C // 64), Tc, Cc, 4 * C, ops.MI_BLOCK_FP16_ATTENTION if half else 0)
    ctx = DeviceBuffer.from_array(oracle.normal(3, B * Tc * Cc))
    kv = DeviceBuffer(ops.block_ctx_kv_bytes(dims))
    ops.block_ctx_kv(bw, dims, ctx, kv)
    synchronize()
    dt, n = (np.float16, B * Tc * C) if half else (np.float32, B * Tc * C)
    for i, name in enumerate(("attn2_k", "attn2_v")):
        out = DeviceBuffer(n * 4)
        if half:
            ops.gemm_nt_q8_0_f16o(ctx, w[name], out, B * Tc, C, Cc)
        else:
            ops.gemm_nt_q8_0(ctx, w[name], out, B * Tc, C, Cc)
        synchronize()
        got = kv.download(dt, n, offset=i * (kv.nbytes // 2))
        assert np.array_equal(got, out.download(dt, n)), name
