"""The one-launch apply and residual of levels 1 to 4 (Replace, Add, residual; Laplace and mass; inner and all DoFs) against
the oracle to 1e-13, and that DoFs the flag leaves out keep their values, on a cube, an octahedron and two cells that
share one face.  src's closure copies are stale (it was uploaded): the kernel reads the owners."""
import numpy as np
import pytest

from helpers import mesh_pair, rel_err, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [("cube", 2), ("gmsh", "regular_octahedron_8el.msh"), ("gmsh", "pyramid_2el.msh")])
@pytest.mark.parametrize("level", [1, 2, 3, 4])
@pytest.mark.parametrize("form", [0, 1])
def test_small_level_apply_matches_oracle(kind, level, form, gpu_ctx, oracle_lib):
    import hyteg_amd as H
    O = oracle_lib
    say(f"[apply cell] {kind} level={level} form={form}")
    om, S = mesh_pair(kind, gpu_ctx)
    xh, yh, bh = np.random.default_rng(level).standard_normal((3, S.owned_count(level)))
    A = (H.P1ConstantLaplaceOperator, H.P1ConstantMassOperator)[form](S, level, level)
    OA, ox = O.Operator(om, level, level, form), O.Function(om, level, level)
    ox.set(level, xh)
    oz = O.Function(om, level, level)
    OA.apply(ox, oz, level, flag=O.ALL)
    product = oz.get(level)
    x, y, b = (H.P1Function(k, S, level, level) for k in "xyb")
    x.upload(level, xh)
    b.upload(level, bh)
    for flag in (H.INNER, H.ALL):
        on = (S.owned_types(level) & flag) != 0
        for what, value in (("replace", product), ("add", yh + product), ("residual", bh - product)):
            y.upload(level, yh)
            if what == "residual":
                A.residual(x, b, y, level, flag)
            else:
                A.apply(x, y, level, flag, H.ADD if what == "add" else H.REPLACE)
            assert rel_err(y.download(level), np.where(on, value, yh)) <= 1e-13, (flag, what)
