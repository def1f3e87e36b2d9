"""The 64x64 GEMM build's 128-k steps and the split layout's whole-block loads:
first, odd and last steps and ragged tiles on the kernel emulator."""
from __future__ import annotations

import json

from test_kemu import BOTH, _run, emulator  # noqa: F401  (fixture)

EMULATED = [dict(M=70, N=70, K=128, cfg="3"), dict(M=65, N=130, K=384, layout="split", front=True, mode=1),
            dict(M=70, N=66, K=640, cfg="3:2"), dict(M=64, N=64, K=192, cfg="3", layout="split"),
            dict(M=200, N=140, K=192, cfg="6", layout="split", front=True), dict(case="gemm_geglu", M=70, F=40, K=384),
            dict(case="gemm_f16a", M=70, N=66, K=384)]


def test_steps_on_emulator(emulator):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    specs = [dict({"case": "gemm_nt"}, schedules=BOTH, **s) for s in EMULATED]
    with ThreadPoolExecutor(8) as ex:
        results = list(ex.map(_run, specs))
    bad = [f"{json.dumps(s)}\n{(r.stdout + r.stderr)[-800:]}" for s, r in zip(specs, results)
           if r.returncode != 0 or r.stdout.count("OK ") != len(BOTH)]
    assert not bad, "\n\n".join(bad)
