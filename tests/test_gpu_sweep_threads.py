"""Two threads sweep different functions of one mesh.  The one-launch sweeps of small levels go through an array of the
level: the launches of a sequence follow each other without another thread's between them, so every result equals, bit
for bit, that of the same sweeps by one thread."""
import threading

import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [1, 3])
def test_threads_sweep_their_own_functions(level, gpu_ctx):
    import hyteg_amd as H
    say(f"[sweep threads] level={level}")
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), 2, 2, 2), gpu_ctx)
    n, rng = S.owned_count(level), np.random.default_rng(level)
    xh, bh = rng.standard_normal((2, 2, n))

    def setup(k):
        A = H.P1ConstantLaplaceOperator(S, 0, level)
        x, b = (H.P1Function(f"{name}{k}", S, 0, level) for name in "xb")
        x.upload(level, xh[k])
        b.upload(level, bh[k])
        return A, x, b

    def work(A, x, b):
        for _ in range(200):
            A.smooth_sor(x, b, 0.9, level, H.INNER)

    expect = []
    for k in range(2):
        state = setup(k)
        work(*state)
        expect.append(state[1].download(level))
    states = [setup(k) for k in range(2)]
    threads = [threading.Thread(target=work, args=s) for s in states]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert np.array_equal(states[k][1].download(level), expect[k])
