"""The few-rows GEMM kernel (M <= 16) at its edges: one row to its last and one
past it (the tiles), columns short of and past a workgroup's 16, one block to
counts that end inside a step of four, more steps than its eight waves
take twice, strides, batch items, modes, both weight layouts, GEGLU, fp16
activations and outputs. On the CPU through the kernel emulator against the
oracle (2e-3 x RMS, the bar of fp16 operands), and bit for bit between the layouts
whatever the alignment of A; on the GPU bit for bit between all entries and forms
(they sum in one order).
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


# One product, every alignment of A: an offset of 1 to 3 floats, rows of every residue of 4, odd batch strides.
BITS = [dict(M=1, N=33, K=96, a_off=1), dict(M=2, N=40, K=1120, a_off=2), dict(M=16, N=20, K=160, pad=1),
        dict(M=5, N=36, K=64, a_off=3, pad=2, batch=3), dict(M=16, N=17, K=1056, pad=3)]


def test_bits_whatever_the_alignment_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict(case="gemm_rows_bits", schedules=BOTH, **s) for s in BITS]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,batch", [(1, 320, 1280, 1), (2, 1280, 1280, 2), (16, 1000, 96, 3), (9, 40, 2816, 2)])
def test_bits_of_every_entry_on_gpu(gpu, oracle, M, N, K, batch):
    """One product through every entry and form that the few-rows kernel serves, bit for bit: batches, strides and
    alignments of A, both layouts, fp16 activations and output, modes 1 and 2, GEGLU."""
    from helpers import q8_weights
    from sdvk_amd import MI_F16, MI_F32, ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    A = oracle.normal(M, batch * M * K).astype(np.float16).astype(np.float32)
    blocks, bias = q8_weights(oracle, 2, N, K), oracle.normal(3, N, 0.0, 0.02)
    C0 = oracle.normal(4, batch * M * N)
    payload, scales = oracle.q8_0_to_split(blocks, N * K)
    dW, dP, dS, dB = (DeviceBuffer.from_array(x) for x in (blocks, payload, scales, bias))

    def out(init=None):
        return DeviceBuffer.from_array(np.zeros(batch * M * N, np.float32) if init is None else init)

    def get(o):
        synchronize()
        return o.download(np.float32, batch * M * N)

    def plain(b):
        o, dA = out(), DeviceBuffer.from_array(A)
        for z in range(batch):
            ops.gemm_nt_q8_0(dA.value + 4 * z * M * K, dW, o.value + 4 * z * M * N, M, N, K, bias=b)
        return get(o)

    want, sums = plain(dB), plain(None)
    stride = dict(batch=batch, sA=M * K, sC=M * N)
    for half in (False, True):
        dA = DeviceBuffer.from_array(A.astype(np.float16) if half else A)
        gemm = ops.gemm_nt_q8_0_f16a if half else ops.gemm_nt_q8_0
        for mode, ref in ((0, want), (1, C0 + sums), (2, C0 + want)):
            o = out(C0)
            gemm(dA, dW, o, M, N, K, bias=dB, mode=mode, **stride)
            assert np.array_equal(get(o), ref), f"mode {mode} half {half}"
        h = DeviceBuffer(batch * M * N * 2)
        for z in range(batch):
            ops.gemm_nt_q8_0_f16o(dA.value + (2 if half else 4) * z * M * K, dW, h.value + 2 * z * M * N, M, N, K,
                                  a_dtype=MI_F16 if half else MI_F32, bias=dB)
        synchronize()
        assert np.array_equal(h.download(np.float16, batch * M * N), want.astype(np.float16))
    for off, pad in ((0, 0), (1, 0), (0, 1), (2, 3)):
        lda, sA = K + pad, M * (K + pad) + pad
        buf = np.zeros(off + batch * sA + K, np.float32)
        for z in range(batch):
            for m in range(M):
                buf[off + z * sA + m * lda:][:K] = A[(z * M + m) * K:][:K]
        dA, o = DeviceBuffer.from_array(buf), out()
        ops.gemm_nt_q8_bias(dA.value + 4 * off, dP, o, dS, dB, M, N, K, lda=lda, batch=batch, sA=sA, sC=M * N)
        assert np.array_equal(get(o), want), f"split layout, offset {off}, rows {pad} apart"
    # GEGLU on the halves of the same columns: value rows, then gate rows
    F, dA = N // 2, DeviceBuffer.from_array(A)
    g, y = DeviceBuffer(M * F * 4), DeviceBuffer(M * F * 4)
    ops.gemm_nt_q8_0_geglu(dA, dW, g, M, F, K, bias=dB)
    dH = DeviceBuffer.from_array(want[:M * N])
    ops.geglu(dH, y, M, F)
    synchronize()
    assert np.array_equal(g.download(np.float32, M * F), y.download(np.float32, M * F)), "GEGLU"


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
