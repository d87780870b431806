"""The backward mode with four, two and one waves to a wave tile, at sizes on
both sides of its rule (block tiles of 32 x 8 pixels: four waves up to 512, or
up to three per light and 2048; two up to 2560) and with blocks whose last wave
tiles hold no pixel; the fused step beside it, on both sides of 4096: against
the FP64 oracle with the adjoint's own bars.
"""
import numpy as np
import pytest

import adjoint_util as A
from test_gpu_adjoint import run_hip, within

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,size", [
    (3, (41, 19)), (16, (403, 405)), (300, (403, 405)), (16, (777, 809)), (900, (777, 809)), (16, (1033, 681)),
    (16, (1604, 1000)), (257, (1604, 1000)),
])
def test_adjoint_matches_fp64(ctx, hlib, n, size):
    print(f"[adjoint share] {size}, {n} lights", flush=True)
    sc, target, _ = A.make_problem(*size, n)
    px = A.decode(sc)
    dpx64, dpos64, dint64 = A.backward64(sc, px, sc.lights, target)
    _, loss64 = A.forward64(sc, px, sc.lights, target)
    r = run_hip(ctx, hlib, sc, target)
    assert abs(r["loss"] - loss64) <= 1e-4 * loss64
    for k in range(5):
        ok, _ = within(r["dpx"][k], dpx64[k], np.abs(dpx64[k]).max())
        assert ok.all(), k
    for a, ref in (("dpos", dpos64), ("dint", dint64)):
        ok, _ = within(r[a], ref, np.abs(ref).max())
        assert ok.all(), a
    for a, b in (("dpx", "b_dpx"), ("dpos", "b_dpos"), ("dint", "b_dint")):
        assert np.all(np.abs(r[a] - r[b]) <= 1e-5 * np.abs(r[a]) + 1e-6 * np.abs(r[a]).max()), a
