"""The tiled NN GEMM with its tiles handed out by XCD (a number of 256-column
tiles that is no multiple of four, B above 2 MB): every tile computed once, at
ragged edges, with and without K splits, in a batch and accumulating. Sums keep
their order whatever the order of the tiles, so a call must agree bit for bit
with the same product over columns padded to four tiles, which takes the grid's
own order."""
import numpy as np
import pytest

from test_kemu import BOTH, _run, emulator  # noqa: F401  (fixture)

CASES = [(130, 260, 2048, 1), (640, 1600, 640, 1), (320, 2304, 320, 2), (129, 60, 8768, 1), (1, 1092, 704, 3)]


def test_on_emulator(emulator):  # noqa: F811
    r = _run(dict(case="gemm_nn", M=130, N=260, K=2048, schedules=BOTH))
    assert r.returncode == 0 and r.stdout.count("OK ") == len(BOTH), (r.stdout + r.stderr)[-800:]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,batch", CASES)
@pytest.mark.parametrize("mode", [0, 1])
def test_bits_of_the_grid_order(gpu, oracle, tune, M, N, K, batch, mode):
    from sdvk_amd import ops
    from sdvk_amd.hip import DeviceBuffer, synchronize

    wide = -(-N // 1024) * 1024  # ldb = ldc: columns N.. are whole tiles of the padded call
    assert -(-N // 256) % 4 and K * N * 4 > 2 << 20
    print(f"[case] nn {M}x{N}x{K} batch {batch} mode {mode}", flush=True)
    payload, scales = oracle.q8_0_to_split(oracle.q8_0_quantize(oracle.normal(1, batch * M * K, 0.0, 0.02)), batch * M * K)
    B, C0 = oracle.normal(2, batch * K * wide), oracle.normal(3, batch * M * wide)
    dq, ds, dB = (DeviceBuffer.from_array(x) for x in (payload, scales, B))

    def call(n, splits):
        tune("nn_splits", splits)
        dC = DeviceBuffer.from_array(C0)
        ws = DeviceBuffer(batch * splits * M * wide * 4) if splits > 1 else None
        ops.gemm_nn_q8(dq, ds, dB, dC, M, n, K, mode=mode, ldb=wide, ldc=wide, batch=batch, sA=M * K, sB=K * wide,
                       sC=M * wide, workspace=ws)
        synchronize()
        return dC.download(np.float32, C0.size).reshape(batch, M, wide)

    for splits in (1, 3):
        got, want = call(N, splits), call(wide, splits)
        assert np.array_equal(got[:, :, :N], want[:, :, :N])
        assert np.array_equal(got[:, :, N:], C0.reshape(batch, M, wide)[:, :, N:])


# Both sides of the rule's edges: unsplit and split, 72 workgroups and more, one row tile, B below and
# above what sends the row tiles to one L2
EDGES = [(320, 2304, 640, 1), (640, 1600, 640, 2), (1280, 400, 2560, 1), (1280, 276, 6464, 1), (100, 1300, 4480, 1),
         (256, 2308, 320, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,batch", EDGES)
def test_bits_at_the_edges_of_the_rule(gpu, oracle, tune, M, N, K, batch):
    test_bits_of_the_grid_order(gpu, oracle, tune, M, N, K, batch, 0)
