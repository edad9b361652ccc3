"""The first call on a mesh: apply, residual and sweeps of the small levels use tables of the whole mesh, which the call
makes.  They are made by the device; loops over the elements on the host took 41 ms for the mesh here (3072
macro-tets, level 4), the rest of a first call is below 1 ms.  The bound lies between, ten times away from either."""
import time

import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


def test_first_call_on_a_large_mesh(gpu_ctx):
    import hyteg_amd as H
    n, level, took = 8, 4, []
    for k in range(3):      # the first also loads the kernels
        S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), n, n, n), gpu_ctx)
        A = H.P1ConstantLaplaceOperator(S, level, level)
        x, y = (H.P1Function(k, S, level, level) for k in "xy")
        x.interpolate_modes(np.array([[1.0, 1, 2, 1]]), level)
        gpu_ctx.synchronize()
        t = time.perf_counter()
        A.apply(x, y, level, H.INNER)
        gpu_ctx.synchronize()
        took.append(time.perf_counter() - t)
        say(f"[first call] {6 * n ** 3} macro-tets, level {level}: {1e3 * took[-1]:.2f} ms")
    assert min(took) < 4e-3
