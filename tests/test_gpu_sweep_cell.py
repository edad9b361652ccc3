"""The one-launch sweep of small levels against the oracle's multicolour sweep: levels 1 (no face or cell interiors) to 4
(the finest), 1 sweep (whose result is copied back) and 2 and 3 in a row with no refresh by the caller, all DoFs and the
inner ones, on a cube, an octahedron and two cells that share one face.  After the sweeps the closure copies are current:
the residual computed from them without a refresh inside a V-cycle is covered by the cycle tests; here the downloaded
micro-vertices, which the library refreshes, equal the owned values.  FP64 to 1e-12 (order of the sums), FP32 to 8e-6
(64 eps: three sweeps of some 30 rounded terms)."""
import numpy as np
import pytest

from helpers import mesh_pair, rel_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [("cube", 2), ("gmsh", "regular_octahedron_8el.msh"), ("gmsh", "pyramid_2el.msh")])
@pytest.mark.parametrize("level", [1, 2, 3, 4])
@pytest.mark.parametrize("sweeps", [1, 2, 3])
def test_small_level_sweeps_match_oracle(kind, level, sweeps, gpu_ctx, oracle_lib):
    import hyteg_amd as H
    O = oracle_lib
    om, S = mesh_pair(kind, gpu_ctx)
    xh, bh = np.random.default_rng(level).standard_normal((2, S.owned_count(level)))
    A, OA = H.P1ConstantLaplaceOperator(S, level, level), O.Operator(om, level, level)
    for precision, flag in ((H.F64, H.INNER), (H.F64, H.ALL), (H.F32, H.INNER)):
        say(f"[sweep cell] {kind} level={level} sweeps={sweeps} precision={precision} flag={flag}")
        x, b = (H.P1Function(k, S, level, level, precision=precision) for k in "xb")
        x.upload(level, xh)
        b.upload(level, bh)
        ox, ob = O.Function(om, level, level), O.Function(om, level, level)
        ox.set(level, xh)
        ob.set(level, bh)
        for _ in range(sweeps):
            A.smooth_sor(x, b, 0.9, level, flag)
            OA.smooth_sor(ox, ob, level, omega=0.9, flag=flag, order=1)
        err = rel_err(x.download(level), ox.get(level))
        say(f"  {err:.2e}")
        assert err <= (1e-12 if precision == H.F64 else 8e-6)
