"""Vector operations on 32 right-hand sides: the parts that a closure range is taken in depend on the number and length of
the ranges."""
import time

import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


def _functions(H, S, level, precision, names):
    return [H.P1Function(k, S, level, level, precision=precision, nrhs=32) for k in names]


def test_short_ranges_are_not_split(gpu_ctx):
    """3072 macro-tets, level 1: 13.9 thousand ranges of a few points.  y += x takes 11 us, in 16 parts each 47 us."""
    import hyteg_amd as H
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), 8, 8, 8), gpu_ctx)
    x, y = _functions(H, S, 1, H.F64, "xy")
    best = 1e9
    for _ in range(5):
        gpu_ctx.synchronize()
        t = time.perf_counter()
        for _ in range(50):
            y.add([1.0], [x], 1, H.INNER)
        gpu_ctx.synchronize()
        best = min(best, (time.perf_counter() - t) / 50)
    say(f"[vector operations] {1e6 * best:.1f} us")
    assert best < 25e-6


@pytest.mark.parametrize("n,level", [(1, 5), (2, 4), (5, 2), (5, 3), (8, 2)])
@pytest.mark.parametrize("precision", [0, 1])
def test_add_and_assign(n, level, precision, gpu_ctx):
    """Parts from 1 to 16.  Quarters and halves of small whole numbers: exact in either precision."""
    import hyteg_amd as H
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), n, n, n), gpu_ctx)
    x, y, z = _functions(H, S, level, precision, "xyz")
    rng = np.random.default_rng(n)
    xh, yh, zh = rng.integers(-1000, 1000, (3, S.owned_count(level), 32)).astype(float)
    x.upload(level, xh), y.upload(level, yh), z.upload(level, zh)
    inner = ((S.owned_types(level) & H.INNER) != 0)[:, None]
    y.add([0.25, 3.0], [x, z], level, H.INNER)
    yh = np.where(inner, yh + 0.25 * xh + 3.0 * zh, yh)
    assert np.array_equal(y.download(level), yh)
    z.assign([0.5], [x], level, H.ALL)
    assert np.array_equal(z.download(level), 0.5 * xh)
