"""The few-rows GEMM kernel (M <= 16) at its edges: one row to its last and one
past it (the tiles), columns short of and past a workgroup's 16, one block to
counts that end inside a step of four, more steps than its eight waves
take twice, strides, batch items, modes, both weight layouts, GEGLU, fp16
activations and outputs. On the CPU through the kernel emulator against the
oracle (2e-3 x RMS, the bar of fp16 operands); on the GPU also bit for bit
between the entries that must agree.
"""
from __future__ import annotations

import json

import numpy as np
import pytest

from test_kemu import BOTH, _run, emulator  # noqa: F401  (fixture)

EMULATED = [
    dict(M=1, N=1, K=32), dict(M=2, N=33, K=96, layout="split", bias_off=1), dict(M=16, N=70, K=1120),
    dict(M=17, N=70, K=96), dict(M=5, N=40, K=1056, mode=1, layout="split", front=True), dict(M=16, N=31, K=64, mode=2),
    dict(M=3, N=36, K=64, batch=3, lda=72, ldc=40, sA=300, sC=130), dict(M=4, N=50, K=100, layout="split"),
    dict(case="gemm_geglu", M=7, F=17, K=96), dict(case="gemm_geglu", M=16, F=40, K=128, ldg=44, front=True),
    dict(case="gemm_f16a", M=9, N=36, K=160, mode=2), dict(case="gemm_f16a", M=2, N=64, K=1280),
    dict(case="gemm_f16o", M=8, N=34, K=96, ldc=36),
    dict(case="block", B=1, T=9, C=64, H=1, Tc=5, Cc=96, F=160, qkv_joint=True, fused=True, half=True),
]


def test_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "gemm_nt"}, schedules=BOTH, **s) if "case" not in s else dict(schedules=BOTH, **s) for s in EMULATED]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 320, 1280), (2, 1280, 1280), (8, 1280, 2816), (16, 1000, 96), (3, 37, 5120)])
def test_on_gpu(gpu, oracle, M, N, K):
    from helpers import assert_parity, q8_weights
    from sdvk_amd import ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    A = oracle.normal(M, M * K)
    blocks = q8_weights(oracle, 2, N, K)
    bias = oracle.normal(3, N, 0.0, 0.02)
    payload, scales = oracle.q8_0_to_split(blocks, N * K)
    dA, dW, dB = DeviceBuffer.from_array(A), DeviceBuffer.from_array(blocks), DeviceBuffer.from_array(bias)
    dP, dS = DeviceBuffer.from_array(payload), DeviceBuffer.from_array(scales)
    dH = DeviceBuffer.from_array(A.astype(np.float16))
    out = [DeviceBuffer(M * N * 4) for _ in range(4)]
    assert ops.gemm_workspace_bytes(M, N, K) == 0
    ops.gemm_nt_q8_0(dA, dW, out[0], M, N, K, bias=dB)
    ops.gemm_nt_q8_0(dA, dW, out[1], M, N, K, bias=dB, workspace=DeviceBuffer(4096))
    ops.gemm_nt_q8_bias(dA, dP, out[2], dS, dB, M, N, K)
    ops.gemm_nt_q8_0_f16a(dH, dW, out[3], M, N, K, bias=dB)
    synchronize()
    got = [o.download(np.float32, M * N) for o in out]
    want = oracle.gemm_nt_q8_0(A, blocks, M, N, K, bias=bias, threads=oracle.max_threads())
    assert_parity(got[0], want, what=f"few rows {M}x{N}x{K}")
    for g in got[1:]:
        assert np.array_equal(got[0], g)
