"""The GEMM's tile rules away from the 1024-pixel shapes, and the 64x64 build's
128-k steps: the planned grids (no workgroup runs), the build's first, odd
and last steps on the kernel emulator, and on the GPU the planned shapes
against the oracle on sampled rows (2e-3 x RMS, the bar of fp16 operands),
the unsplit ones bit for bit against another tile build.
"""
from __future__ import annotations

import json

import numpy as np
import pytest

from test_kemu import BOTH, _run, emulator  # noqa: F401  (fixture)

ROUTES = [
    ["gemm", [576, 1280, 1280], [180, 1, 1], 256], ["gemm_ws", [576, 1280, 1280], [180, 1, 1], 256],
    ["gemm", [1600, 1280, 1280], [500, 1, 1], 256], ["gemm", [1976, 1280, 1280], [160, 1, 1], 512],
    ["gemm", [3952, 640, 640], [155, 1, 1], 512], ["gemm", [7904, 640, 2560], [155, 1, 1], 512],
    ["gemm_ws", [576, 1280, 5120], [50, 5, 1], 512], ["gemm_ws", [988, 1280, 5120], [80, 3, 1], 512],
    ["gemm_ws", [1152, 1280, 5120], [50, 5, 1], 512], ["gemm_ws", [1024, 640, 2560], [160, 1, 1], 256],
    ["gemm_ws", [4608, 640, 2560], [180, 1, 1], 512], ["gemm_ws", [308, 640, 2048], [50, 4, 1], 256],
]
# Few tiles: K parts of 64x64 as long as the 128x128 tiles' parts cost more, in counts that whole
# steps reach and that the reduce pass loads at once
FEW_TILES = [
    ["gemm_ws", [77, 768, 3072], [24, 8, 1], 256], ["gemm_ws", [154, 768, 3072], [36, 4, 1], 256],
    ["gemm_ws", [77, 1280, 5120], [40, 4, 1], 256], ["gemm_ws", [154, 1280, 5120], [60, 4, 1], 256],
    ["gemm_ws", [308, 768, 3072], [60, 4, 1], 256], ["gemm_ws", [17, 1280, 5120], [20, 8, 1], 256],
    ["gemm_ws", [154, 640, 2560], [30, 8, 1], 256], ["gemm_ws", [256, 640, 2560], [40, 4, 1], 256],
    ["gemm_ws", [512, 640, 2560], [80, 3, 1], 256], ["gemm_ws", [256, 1280, 5120], [20, 8, 1], 512],
    ["gemm_ws", [154, 1280, 1280], [60, 4, 1], 256], ["gemm_ws", [77, 640, 1280], [20, 4, 1], 256],
    ["gemm_ws", [77, 640, 768], [20, 4, 1], 256], ["gemm_ws", [231, 1280, 1280], [80, 3, 1], 256],
    ["gemm_ws", [17, 640, 2048], [10, 8, 1], 256], ["gemm_ws", [308, 1280, 1280], [100, 2, 1], 256],
]
# K % 64 != 0 runs on 64x64 tiles alone: parts by their count, not by the 128x128 tiles'
GENERAL = [
    ["gemm_ws", [988, 640, 2592], [160, 3, 1], 256], ["gemm_ws", [768, 640, 5152], [120, 4, 1], 256],
    ["gemm_ws", [1440, 1280, 5152], [460, 1, 1], 256], ["gemm_ws", [154, 640, 2592], [30, 8, 1], 256],
    ["gemm_ws", [154, 1280, 3104], [60, 4, 1], 256], ["gemm_ws", [768, 1280, 5152], [240, 2, 1], 256],
]
COUNTS = [(M, N, K) for M in (17, 77, 154, 231, 308, 512, 576, 988) for N, K in (
    (768, 768), (768, 3072), (1280, 1280), (1280, 5120), (640, 640), (640, 2560), (1280, 320), (1280, 2816), (320, 1280),
    (640, 96), (640, 160), (640, 2592), (1280, 11200))]
EMULATED = [dict(M=70, N=70, K=128, cfg="3"), dict(M=65, N=130, K=384, layout="split", front=True, mode=1),
            dict(M=70, N=66, K=640, cfg="3:2"), dict(M=64, N=64, K=192, cfg="3", layout="split"),
            dict(M=200, N=140, K=192, cfg="6", layout="split", front=True), dict(case="gemm_geglu", M=70, F=40, K=384),
            dict(case="gemm_f16a", M=70, N=66, K=384)]


def test_plans(emulator):  # noqa: F811
    r = _run({"case": "routing", "table": ROUTES})
    assert r.returncode == 0 and "OK routing" in r.stdout, (r.stdout + r.stderr)[-2000:]


@pytest.mark.parametrize("table", ["FEW_TILES", "GENERAL"])
def test_split_plans(emulator, table):  # noqa: F811
    r = _run({"case": "routing", "table": globals()[table]})
    assert r.returncode == 0 and "OK routing" in r.stdout, (r.stdout + r.stderr)[-2000:]


def test_split_counts_launched_as_planned(emulator):  # noqa: F811
    r = _run({"case": "split_counts", "shapes": COUNTS})
    assert r.returncode == 0 and "OK split_counts" in r.stdout, (r.stdout + r.stderr)[-2000:]


# Split builds of the plans on few tiles: 64-k steps although K % 128 == 0, 128-k steps, an odd last part
SPLITS = [dict(M=70, N=66, K=1280), dict(M=77, N=70, K=768, mode=1), dict(M=65, N=130, K=2560, layout="split", mode=2),
          dict(M=40, N=64, K=2816, front=True), dict(M=70, N=66, K=640, cfg="3:5"), dict(case="gemm_f16a", M=70, N=66, K=1280)]


def test_splits_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "gemm_nt"}, schedules=BOTH, **s) for s in SPLITS]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


def test_steps_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "gemm_nt"}, schedules=BOTH, **s) for s in EMULATED]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,split", [(77, 768, 3072, True), (154, 1280, 1280, True), (231, 1280, 1280, True),
                                         (77, 1280, 2816, True), (17, 640, 2560, True),
                                         (988, 640, 2592, True), (576, 1280, 5120, True), (988, 1280, 5120, True), (1152, 1280, 5120, True),
                                         (1152, 1280, 1280, False), (3952, 640, 640, False), (7904, 640, 2560, False)])
def test_planned_shapes(gpu, oracle, tune, M, N, K, split):
    from helpers import REL_RMS_TOL, err_vs_rms, q8_weights
    from sdvk_amd import ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    A, blocks = oracle.normal(1, M * K), q8_weights(oracle, 2, N, K)
    dA, dW, dC = DeviceBuffer.from_array(A), DeviceBuffer.from_array(blocks), DeviceBuffer(M * N * 4)
    nws = ops.gemm_workspace_bytes(M, N, K)
    assert (nws > 0) == split
    ops.gemm_nt_q8_0(dA, dW, dC, M, N, K, workspace=DeviceBuffer(nws) if nws else None)
    synchronize()
    got = dC.download(np.float32, M * N).reshape(M, N)
    rows = np.unique(np.concatenate([[0, M - 1], np.random.default_rng(M).integers(0, M, 48)]))
    assert err_vs_rms(got[rows], oracle.gemm_rows(A, blocks, M, N, K, rows, threads=oracle.max_threads())) <= REL_RMS_TOL
    if not split:
        tune("gemm_cfg", "5")
        ops.gemm_nt_q8_0(dA, dW, dC, M, N, K)
        synchronize()
        assert np.array_equal(dC.download(np.float32, M * N).reshape(M, N), got)
