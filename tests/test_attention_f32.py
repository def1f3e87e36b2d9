"""The pipelined fp32 attention kernel at the sizes where it can go wrong: one
and two key groups (512 keys is where the second may start), partial key
tiles and sub-tiles, a single key, head dims below 64, masks, rows of
several strides, a negative scale, outlying keys (the rescale), both P
precisions and output types. On the CPU through the kernel emulator, on the
GPU through the C-ABI, against the oracle.

Bars: P in two fp16 parts (fp32 outputs): the reference test's own 2e-5
relative (tests/fused_attn_test.cpp:118-126), taken of the output's RMS; P as
one fp16 value: its rounding besides, at most 2^-11 of each weight p in the
numerator and in the row sum, so 2^-11 (sum p |v| + |o|) per output (emulator
cases: 2e-3 x RMS, the common bar).
"""
from __future__ import annotations

import json
import sys

import numpy as np
import pytest

from test_kemu import BOTH, KEMU, _run, emulator  # noqa: F401  (fixture)

EMULATED = [
    # two key groups: odd and even trip counts, a last tile / sub-tile of one key, a trip past the keys
    dict(Tq=130, Tk=512, C=64, heads=1, precision=0, tol=2e-5), dict(Tq=33, Tk=577, C=128, heads=2, precision=0, tol=2e-5),
    dict(Tq=64, Tk=641, C=40, heads=1), dict(Tq=200, Tk=640, C=64, heads=1, causal=True, precision=0, tol=2e-5),
    dict(batch=2, Tq=40, Tk=700, C=64, heads=1, kv_len=[65, 1], precision=0, tol=2e-5),
    dict(Tq=64, Tk=520, C=64, heads=1, outliers=[5, 70, 511]), dict(Tq=40, Tk=530, C=64, heads=1, f16_out=True),
    # one group: a key, a sub-tile and one more, a tile and one more, masks, the unstaged output store
    dict(Tq=5, Tk=1, C=64, heads=1, precision=0, tol=2e-5), dict(Tq=70, Tk=33, C=16, heads=2, precision=0, tol=2e-5),
    dict(Tq=70, Tk=65, C=64, heads=1, f16_out=True, front=True), dict(batch=2, Tq=33, Tk=97, C=64, heads=1, kv_len=[0, 32]),
    dict(Tq=131, Tk=131, C=64, heads=1, causal=True, front=True, precision=0, tol=2e-5),
    dict(Tq=64, Tk=192, C=64, heads=1, outliers=[5, 66, 134], direct_store=True),
]


def test_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "attention"}, schedules=BOTH, **s) for s in EMULATED]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


# First keys far below the rest, in one and two sub-tiles, one and two key groups: the scores
# that follow are taken before the running max leaves its first value and must keep
# fp32's bits, so the plain bar holds whatever the distance.
LOW = [dict(Tq=40, Tk=96, C=64, heads=1, low=[32, 1000]), dict(Tq=33, Tk=200, C=128, heads=2, low=[40, 100]),
       dict(Tq=40, Tk=600, C=64, heads=1, low=[32, 5000])]


def test_low_first_keys_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "attention"}, schedules=BOTH, precision=0, tol=2e-5, **s) for s in LOW]
    with ThreadPoolExecutor(4) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("Tk,n,d", [(96, 32, 1000.0), (200, 40, 100.0), (600, 32, 5000.0), (1024, 64, 300.0)])
def test_low_first_keys_on_gpu(gpu, oracle, Tk, n, d):
    from sdvk_amd import MI_F32, ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    q, k, v = (oracle.normal(i, t * 64).reshape(t, 64) for i, t in ((1, 130), (2, Tk), (3, Tk)))
    q[:, 0], k[:, 0], k[:n, 0] = 1.0, 0.0, -8.0 * d
    s = q.astype(np.float64) @ k.astype(np.float64).T / 8.0
    p = np.exp(s - s.max(-1, keepdims=True))
    want = p @ v.astype(np.float64) / p.sum(-1, keepdims=True)
    dq, dk, dv, do = (DeviceBuffer.from_array(x) for x in (q, k, v, np.zeros_like(q)))
    ops.fused_attention_ex(dq, dk, dv, do, batch=1, Tq=130, Tk=Tk, C=64, heads=1, in_dtype=MI_F32, out_dtype=MI_F32)
    synchronize()
    got = do.download(np.float32, q.size).reshape(q.shape)
    assert np.abs(got - want).max() <= 2e-5 * np.sqrt(np.mean(want ** 2))


# Keys that end with a tile's first sub-tile (the loop leaves there) and one past it, in one and two
# key groups, by the mask of a causal launch, and by the lengths of a batch
ENDS = [dict(Tq=32, Tk=32, C=64, heads=1), dict(Tq=40, Tk=96, C=16, heads=2), dict(Tq=32, Tk=64, C=64, heads=1, causal=True),
        dict(Tq=160, Tk=160, C=64, heads=1, causal=True), dict(Tq=20, Tk=544, C=64, heads=1), dict(Tq=20, Tk=545, C=64, heads=1),
        dict(Tq=20, Tk=608, C=64, heads=1), dict(Tq=20, Tk=609, C=64, heads=1), dict(Tq=150, Tk=700, C=64, heads=1, causal=True),
        dict(batch=3, Tq=9, Tk=600, C=64, heads=1, kv_len=[32, 0, 33]), dict(batch=2, Tq=9, Tk=90, C=64, heads=1, kv_len=[64, 65])]


def test_ends_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "attention"}, schedules=BOTH, precision=0, tol=2e-5, **s) for s in ENDS]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Tq,Tk,C,heads,causal", [
    (1, 7, 7, 80, 5, False), (2, 26, 26, 128, 8, False), (1, 64, 64, 128, 2, True), (1, 96, 96, 64, 1, False),
    (1, 160, 160, 640, 10, True), (1, 300, 544, 640, 10, False), (1, 300, 609, 640, 10, False)])
def test_ends_on_gpu(gpu, oracle, B, Tq, Tk, C, heads, causal):
    test_on_gpu(gpu, oracle, B, Tq, Tk, C, heads, causal, 0, 0.0)


@pytest.mark.parametrize("Tk", [2, 3, 8])
def test_no_product_of_residuals_left_out_on_emulator(emulator, Tk):  # noqa: F811
    r = _run(dict(case="attention_residuals", Tk=Tk, schedules=BOTH))
    assert r.returncode == 0 and r.stdout.count("OK ") == len(BOTH), (r.stdout + r.stderr)[-800:]


@pytest.mark.gpu
@pytest.mark.parametrize("Tk", [2, 3])
def test_no_product_of_residuals_left_out_on_gpu(gpu, Tk):
    """A few keys: over many the MFMA's own accumulation has a bias of this size."""
    sys.path.insert(0, str(KEMU))
    from cases import residual_bias, residual_inputs
    from sdvk_amd import MI_F32, ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    q, k, v = residual_inputs(np.random.default_rng(Tk), 128, Tk)
    dq, dk, dv, do = (DeviceBuffer.from_array(x) for x in (q, k, v, np.zeros_like(q)))
    ops.fused_attention_ex(dq, dk, dv, do, batch=1, Tq=128, Tk=Tk, C=64, heads=1, in_dtype=MI_F32, out_dtype=MI_F32)
    synchronize()
    e = residual_bias(do.download(np.float32, q.size).reshape(q.shape).astype(np.float64), q, k, v)
    print(f"[case] {Tk} keys: mean error {e:.2e}", flush=True)
    assert abs(e) <= 2.0 ** -23


@pytest.mark.gpu
@pytest.mark.parametrize("B,Tq,Tk,C,heads,causal,pad,scale", [
    (1, 129, 512, 640, 10, False, 0, 0.0), (1, 300, 577, 640, 10, False, 4, 0.0), (1, 257, 700, 320, 5, True, 0, 0.0),
    (2, 4096, 96, 640, 10, False, 0, 0.0), (2, 2100, 530, 640, 10, False, 0, 0.05), (1, 100, 640, 128, 2, False, 0, -0.125),
    (2, 70, 77, 40, 1, False, 8, 0.0), (1, 33, 31, 16, 2, False, 0, 0.0), (3, 77, 77, 768, 12, True, 0, 0.0)])
def test_on_gpu(gpu, oracle, B, Tq, Tk, C, heads, causal, pad, scale):
    from sdvk_amd import MI_ATTN_PREC_FP16, MI_F32, ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    ld = C + pad
    q, k, v = (oracle.normal(i, B * t * ld).reshape(B, t, ld) for i, t in ((1, Tq), (2, Tk), (3, Tk)))
    qd, kd, vd = (x[:, :, :C].astype(np.float64).reshape(B, -1, heads, C // heads).transpose(0, 2, 1, 3) for x in (q, k, v))
    s = np.einsum("bhqd,bhkd->bhqk", qd, kd) * (scale or 1.0 / np.sqrt(C // heads))
    if causal:
        s = np.where(np.arange(Tk)[None, :] > np.arange(Tq)[:, None], -np.inf, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want, spread = ((p @ x).transpose(0, 2, 1, 3).reshape(B, Tq, C) for x in (vd, np.abs(vd)))
    bar = 2e-5 * np.sqrt(np.mean(want ** 2))
    dq, dk, dv = (DeviceBuffer.from_array(x) for x in (q, k, v))
    for precision in (0, MI_ATTN_PREC_FP16):
        do = DeviceBuffer.from_array(np.full(B * Tq * ld, 7.0, np.float32))
        ops.fused_attention_ex(dq, dk, dv, do, batch=B, Tq=Tq, Tk=Tk, C=C, heads=heads, causal=causal, in_dtype=MI_F32,
                               out_dtype=MI_F32, ldq=ld, ldk=ld, ldv=ld, ldo=ld, scale=scale, precision=precision)
        synchronize()
        got = do.download(np.float32, B * Tq * ld).reshape(B, Tq, ld)
        assert np.all(got[:, :, C:] == 7.0)
        e = np.abs(got[:, :, :C] - want) / (bar + (2.0 ** -11 * (spread + np.abs(want)) if precision else 0.0))
        print(f"[case] {B}x{heads}x{Tq}x{Tk} precision {precision}: {e.max():.2f} of the bar", flush=True)
        assert e.max() <= 1.0


@pytest.mark.gpu
def test_more_workgroups_than_a_1d_launch(gpu):
    """2^24 and more (batch, head) pairs: 256 threads each no longer fit one grid dimension. One key: out = v."""
    from sdvk_amd import MI_F32, ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    B, heads, hd = 65535, 257, 8
    v = np.arange(B * heads * hd, dtype=np.float32) % 8191
    dv = DeviceBuffer.from_array(v)
    dq, do = DeviceBuffer.from_array(np.ones_like(v)), DeviceBuffer(v.nbytes)
    ops.fused_attention_ex(dq, dq, dv, do, batch=B, Tq=1, Tk=1, C=heads * hd, heads=heads, in_dtype=MI_F32,
                           out_dtype=MI_F32)
    synchronize()
    # values below 2^13 are whole: one key's weight is 1, hi + lo carries 2^-22 of a value
    assert np.abs(do.download(np.float32, v.size) - v).max() <= 8191 * 2.0 ** -21
