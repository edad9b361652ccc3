"""Sweeps of small levels by separate launches, a workgroup per face and per cell, on meshes of many cells.  Their LDS and
workgroups have to be those of the level: with level 5's, few of them fitted a CU and a sweep at level 3 on 10368
macro-tets took 4.1 times an apply's time, now 2.3."""
import time

import numpy as np
import pytest

from helpers import rel_err, say

pytestmark = pytest.mark.gpu


def test_sweep_against_apply(gpu_ctx):
    import hyteg_amd as H
    n, level = 12, 3
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), n, n, n), gpu_ctx)
    A = H.P1ConstantLaplaceOperator(S, level, level)
    x, b, y = (H.P1Function(k, S, level, level) for k in "xby")
    x.interpolate_modes(np.array([[1.0, 1, 2, 1]]), level)
    best = {}
    for _ in range(5):
        for name, call in (("sweep", lambda: A.smooth_sor(x, b, 1.0, level, H.INNER)),
                           ("apply", lambda: A.apply(x, y, level, H.INNER))):
            gpu_ctx.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                call()
            gpu_ctx.synchronize()
            best[name] = min(best.get(name, 1e9), (time.perf_counter() - t) / 20)
    say(f"[sweep of many cells] {({k: round(1e6 * v, 1) for k, v in best.items()})} us")
    assert best["sweep"] < 3.2 * best["apply"]


@pytest.mark.parametrize("level", [2, 3, 4, 5])
@pytest.mark.parametrize("precision", [0, 1])
def test_sweeps_match_oracle(level, precision, gpu_ctx, oracle_lib):
    """A row of 258 tetrahedra, each sharing a face with the next, forward and backward; FP64 to 1e-12, FP32 to 64 eps (two
    sweeps of some 30 rounded terms)."""
    import hyteg_amd as H
    O = oracle_lib
    t = np.arange(261)
    X = np.stack([np.cos(2.3 * t), np.sin(2.3 * t), 0.35 * t], axis=1)
    C = np.stack([t[:-3], t[1:-2], t[2:-1], t[3:]], axis=1).astype(np.int32)
    S = H.PrimitiveStorage(H.MeshInfo.fromArrays(X, C), gpu_ctx)
    om = O.Mesh.from_arrays(X, C)
    xh, bh = np.random.default_rng(level).standard_normal((2, S.owned_count(level)))
    A, OA = H.P1ConstantLaplaceOperator(S, level, level), O.Operator(om, level, level)
    x, b = (H.P1Function(k, S, level, level, precision=precision) for k in "xb")
    ox, ob = O.Function(om, level, level), O.Function(om, level, level)
    x.upload(level, xh), b.upload(level, bh), ox.set(level, xh), ob.set(level, bh)
    A.smooth_sor(x, b, 0.9, level, H.ALL)
    A.smooth_sor_backwards(x, b, 0.9, level, H.ALL)
    OA.smooth_sor(ox, ob, level, omega=0.9, flag=O.ALL, order=1)
    OA.smooth_sor_backward(ox, ob, level, omega=0.9, flag=O.ALL, order=1)
    err = rel_err(x.download(level), ox.get(level))
    say(f"[sweep of many cells] level={level} precision={precision}: {err:.2e}")
    assert err <= (1e-12 if precision == H.F64 else 8e-6)
