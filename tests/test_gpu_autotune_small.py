"""The autotuner on a small level, where a sweep is one launch for all primitives unless the fused cell phase is selected:
what it compares has to be whole sweeps.  Two of them take at least as long as 0.6 times two calls of one sweep
each (a call copies its result back as well); the cell phases alone that it timed before took a third of that."""
import time

import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [3, 4])
def test_small_level_compares_whole_sweeps(level, gpu_ctx):
    import hyteg_amd as H
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), 2, 2, 2), gpu_ctx)
    A = H.P1ConstantLaplaceOperator(S, level, level)
    x, b = (H.P1Function(k, S, level, level) for k in "xb")
    x.interpolate_modes(np.array([[1.0, 1, 2, 1]]), level)

    def sweep_time():
        best = 1e9
        for _ in range(5):
            gpu_ctx.synchronize()
            t = time.perf_counter()
            for _ in range(100):
                A.smooth_sor(x, b, 1.0, level, H.INNER)
            gpu_ctx.synchronize()
            best = min(best, (time.perf_counter() - t) / 100)
        return 1e3 * best

    before = sweep_time()
    rep = S.autotune(level, reps=20)
    passes, fused = rep[-4:-2]
    tile, bits = S.get_cell_sor_setting(level)
    say(f"[autotune] level {level}: one sweep {before:.4f} ms, two without and with the fused phase {passes:.4f} {fused:.4f}, "
        f"tile {tile} bits {bits}")
    assert passes > 0.6 * 2 * before
    if not (tile and bits & 1):
        assert sweep_time() < 1.5 * before
