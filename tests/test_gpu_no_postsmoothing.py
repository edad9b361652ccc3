"""Cycles without post-smoothing: the coarse x that is prolongated, and the one a W-cycle visits again, then ends with a
prolongation, which leaves its closure copies behind.  V(2,0), V(1,0), V(0,1) and W(2,0) against the oracle's cycles."""
import numpy as np
import pytest

from helpers import mesh_pair, rel_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [("cube", 2), ("gmsh", "regular_octahedron_8el.msh")])
@pytest.mark.parametrize("level", [3, 6])
@pytest.mark.parametrize("pre,post,wcycle", [(2, 0, 0), (1, 0, 0), (0, 1, 0), (2, 0, 1)])
def test_cycles_match_oracle(kind, level, pre, post, wcycle, gpu_ctx, oracle_lib):
    import hyteg_amd as H
    O = oracle_lib
    say(f"[no post-smoothing] {kind} level={level} ({pre},{post}) wcycle={wcycle}")
    om, S = mesh_pair(kind, gpu_ctx)
    bh = np.random.default_rng(level).standard_normal(om.owned_count(level))
    bh[(S.owned_types(level) & H.INNER) == 0] = 0.0
    A, OA = H.P1ConstantLaplaceOperator(S, 0, level), O.Operator(om, 0, level)
    x, b = H.P1Function("x", S, 0, level), H.P1Function("b", S, 0, level)
    ox, ob = O.Function(om, 0, level), O.Function(om, 0, level)
    b.upload(level, bh)
    ob.set(level, bh)
    gmg = H.GeometricMultigridSolver(S, H.SORSmoother(1.0), H.CGSolver(S, 0, 0), H.P1toP1LinearRestriction(),
                                     H.P1toP1LinearProlongation(), 0, level, pre, post, cycleType=wcycle)
    og = O.GMG(om, 0, level, pre, post, 1.0, 1, wcycle=wcycle)
    for cycle in range(2):
        gmg.solve(A, x, b, level)
        og.solve(OA, ox, ob, level)
        err = rel_err(x.download(level), ox.get(level))
        say(f"  cycle {cycle}: {err:.2e}")
        assert err <= 1e-11, cycle
