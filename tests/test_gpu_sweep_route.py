"""Forward sweeps of a small level on many macro-cells must not take the form in which every cell recomputes what surrounds
it.  A backward sweep always runs as separate launches and does the same work, with a refresh more: at 3072 macro-tets
and level 4 a forward sweep by separate launches takes 0.84 (FP32) and 0.87 (FP64) of its time, the one-launch
form 1.36 and 1.29."""
import time

import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
def test_forward_sweep_of_many_cells(precision, gpu_ctx):
    import hyteg_amd as H
    n, level = 8, 4
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), n, n, n), gpu_ctx)
    A = H.P1ConstantLaplaceOperator(S, level, level)
    x, b = (H.P1Function(k, S, level, level, precision=precision) for k in "xb")
    x.interpolate_modes(np.array([[1.0, 1, 2, 1]]), level)
    best = {}
    for _ in range(5):
        for sweep in (A.smooth_sor, A.smooth_sor_backwards):
            gpu_ctx.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                sweep(x, b, 1.0, level, H.INNER)
            gpu_ctx.synchronize()
            best[sweep.__name__] = min(best.get(sweep.__name__, 1e9), (time.perf_counter() - t) / 20)
    say(f"[sweep route] precision={precision} {({k: round(1e6 * v, 1) for k, v in best.items()})} us")
    assert best["smooth_sor"] < 1.1 * best["smooth_sor_backwards"]


@pytest.mark.parametrize("cells", [250, 258, 510, 516])
@pytest.mark.parametrize("level", [1, 2, 3])
def test_sweeps_on_both_sides_of_the_limits(cells, level, gpu_ctx, oracle_lib):
    """A row of tetrahedra, each sharing a face with the next, so that any number of cells can be had."""
    import hyteg_amd as H
    O = oracle_lib
    t = np.arange(cells + 3)
    X = np.stack([np.cos(2.3 * t), np.sin(2.3 * t), 0.35 * t], axis=1)
    C = np.stack([t[:-3], t[1:-2], t[2:-1], t[3:]], axis=1).astype(np.int32)
    S = H.PrimitiveStorage(H.MeshInfo.fromArrays(X, C), gpu_ctx)
    om = O.Mesh.from_arrays(X, C)
    A, OA = H.P1ConstantLaplaceOperator(S, level, level), O.Operator(om, level, level)
    xh, bh = np.random.default_rng(level).standard_normal((2, S.owned_count(level)))
    x, b = (H.P1Function(k, S, level, level) for k in "xb")
    ox, ob = O.Function(om, level, level), O.Function(om, level, level)
    x.upload(level, xh), b.upload(level, bh), ox.set(level, xh), ob.set(level, bh)
    for _ in range(3):
        A.smooth_sor(x, b, 0.9, level, H.ALL)
        OA.smooth_sor(ox, ob, level, omega=0.9, flag=O.ALL, order=1)
    got, ref = x.download(level), ox.get(level)
    err = np.abs(got - ref).max() / np.abs(ref).max()
    say(f"[sweep route] {cells} cells level={level}: {err:.2e}")
    assert err <= 1e-12
