"""Sweeps on 32 right-hand sides on meshes of many cells: which classes run in one launch each depends on the number of
workgroups, and their LDS on the level."""
import time

import numpy as np
import pytest

from helpers import rel_err, say

pytestmark = pytest.mark.gpu


def test_sweep_against_apply(gpu_ctx):
    """3072 macro-tets, level 3, FP64: a sweep takes 1.8 times an apply's time; with every class in one launch and the
    LDS arrays of the finest level 3.6 times."""
    import hyteg_amd as H
    n, level = 8, 3
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), n, n, n), gpu_ctx)
    A = H.P1ConstantLaplaceOperator(S, level, level)
    x, b, y = (H.P1Function(k, S, level, level, nrhs=32) for k in "xby")
    x.interpolate_modes(np.tile([[[1.0, 1, 2, 1]]], (32, 1, 1)), level)
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
    say(f"[multi SOR, many cells] {({k: round(1e6 * v, 1) for k, v in best.items()})} us")
    assert best["sweep"] < 2.6 * best["apply"]


@pytest.mark.parametrize("cells,level", [(400, 1), (450, 1), (60, 4), (300, 4), (450, 2), (30, 5), (130, 5), (450, 3)])
@pytest.mark.parametrize("precision", [0, 1])
def test_columns_match_oracle(cells, level, precision, gpu_ctx, oracle_lib):
    """A row of tetrahedra, each sharing a face with the next; sizes on both sides of the limits of the edges (level 1) and
    of the faces (levels 4 and 5).  Two sweeps; FP64 to 1e-12 (the sums' order differs), FP32 to 64 eps (some 30 terms
    each)."""
    import hyteg_amd as H
    O = oracle_lib
    t = np.arange(cells + 3)
    X = np.stack([np.cos(2.3 * t), np.sin(2.3 * t), 0.35 * t], axis=1)
    C = np.stack([t[:-3], t[1:-2], t[2:-1], t[3:]], axis=1).astype(np.int32)
    S = H.PrimitiveStorage(H.MeshInfo.fromArrays(X, C), gpu_ctx)
    om = O.Mesh.from_arrays(X, C)
    xh, bh = np.random.default_rng(level).standard_normal((2, S.owned_count(level), 32))
    A, OA = H.P1ConstantLaplaceOperator(S, level, level), O.Operator(om, level, level)
    x, b = (H.P1Function(k, S, level, level, precision=precision, nrhs=32) for k in "xb")
    x.upload(level, xh)
    b.upload(level, bh)
    for _ in range(2):
        A.smooth_sor(x, b, 0.9, level, H.ALL)
    got = x.download(level)
    for col in (0, 7, 8, 31):
        ox, ob = O.Function(om, level, level), O.Function(om, level, level)
        ox.set(level, np.ascontiguousarray(xh[:, col]))
        ob.set(level, np.ascontiguousarray(bh[:, col]))
        for _ in range(2):
            OA.smooth_sor(ox, ob, level, omega=0.9, flag=O.ALL, order=1)
        err = rel_err(got[:, col], ox.get(level))
        say(f"[multi SOR, many cells] {cells} cells level={level} precision={precision} column {col}: {err:.2e}")
        assert err <= (1e-12 if precision == H.F64 else 8e-6), col
