"""Forward SOR sweeps on 32 interleaved right-hand sides (one launch per primitive class on small levels) against the
oracle's multicolour sweep, column by column: levels without face and cell interiors (1), with one cell point (2), the
finest level of the one-launch cells (5) and the first of the colour passes (6).  Two sweeps follow each other without
a refresh by the caller, so stale closure copies would show.  FP64 to 1e-12 (the sums' order differs); FP32 to
64 eps = 8e-6 of the largest value: two sweeps of at most some 30 terms each, every term rounded to 2^-24 relative."""
import numpy as np
import pytest

from helpers import mesh_pair, rel_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [("cube", 2), ("gmsh", "regular_octahedron_8el.msh"), ("gmsh", "pyramid_2el.msh")])
@pytest.mark.parametrize("level", [1, 2, 3, 5, 6])
@pytest.mark.parametrize("precision", [0, 1])
def test_columns_of_a_sweep_match_oracle(kind, level, precision, gpu_ctx, oracle_lib):
    import hyteg_amd as H
    O = oracle_lib
    say(f"[multi SOR] {kind} level={level} precision={precision}")
    om, S = mesh_pair(kind, gpu_ctx)
    n, rng = S.owned_count(level), np.random.default_rng(level)
    xh, bh = rng.standard_normal((2, n, 32))
    A, OA = H.P1ConstantLaplaceOperator(S, level, level), O.Operator(om, level, level)
    x, b = (H.P1Function(k, S, level, level, precision=precision, nrhs=32) for k in "xb")
    x.upload(level, xh)
    b.upload(level, bh)
    for _ in range(2):
        A.smooth_sor(x, b, 0.9, level, H.INNER)
    got = x.download(level)
    for col in (0, 7, 8, 31):
        ox, ob = O.Function(om, level, level), O.Function(om, level, level)
        ox.set(level, np.ascontiguousarray(xh[:, col]))
        ob.set(level, np.ascontiguousarray(bh[:, col]))
        for _ in range(2):
            OA.smooth_sor(ox, ob, level, omega=0.9, flag=O.INNER, order=1)
        err = rel_err(got[:, col], ox.get(level))
        say(f"  column {col}: {err:.2e}")
        assert err <= (1e-12 if precision == H.F64 else 8e-6), col
