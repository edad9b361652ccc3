"""A mesh with a node that no tetrahedron uses (as mesh generators leave them): its vertex is an unknown like any other, with
an empty stencil row.  Apply, residual and sweeps give it what such a row gives on every level, the small ones (one
workgroup per macro-cell) included: A x = 0, y + A x = y, b - A x = b exactly, and a sweep leaves it alone.  The
other values equal those of the mesh without the node to 1e-13 (the sums are the same; their order may differ)."""
import numpy as np
import pytest

from helpers import rel_err, say

pytestmark = pytest.mark.gpu

X = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1], [1, 1, 1], [-1, 0.5, 0.2]], dtype=float)
CELLS = np.array([[0, 1, 2, 3], [1, 2, 3, 4], [0, 2, 3, 5]], dtype=np.int32)


@pytest.mark.parametrize("level", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("precision", [0, 1])
def test_unused_node_has_an_empty_row(level, precision, gpu_ctx):
    import hyteg_amd as H
    say(f"[lone vertex] level={level} precision={precision}")
    lone = len(X)
    S = H.PrimitiveStorage(H.MeshInfo.fromArrays(np.vstack([X, [[3.0, 3.0, 3.0]]]), CELLS), gpu_ctx)
    S0 = H.PrimitiveStorage(H.MeshInfo.fromArrays(X, CELLS), gpu_ctx)
    n = S.owned_count(level)
    assert n == S0.owned_count(level) + 1
    rest = np.arange(n) != lone
    xh, yh, bh = np.random.default_rng(level).standard_normal((3, n)).astype(np.float32).astype(np.float64)

    def results(S, keep):
        A = H.P1ConstantLaplaceOperator(S, level, level)
        x, y, b = (H.P1Function(k, S, level, level, precision=precision) for k in "xyb")
        x.upload(level, xh[keep])
        b.upload(level, bh[keep])
        out = {}
        for what in ("replace", "add", "residual"):
            y.upload(level, yh[keep])
            if what == "residual":
                A.residual(x, b, y, level, H.ALL)
            else:
                A.apply(x, y, level, H.ALL, H.ADD if what == "add" else H.REPLACE)
            out[what] = y.download(level)
        for k in range(3):
            A.smooth_sor(x, b, 0.9, level, H.INNER)
            out[f"sweep {k}"] = x.download(level)
        return out

    got, ref = results(S, np.ones(n, bool)), results(S0, rest)
    alone = {"replace": 0.0, "add": yh[lone], "residual": bh[lone]}
    for what, value in got.items():
        if level > 0 or not what.startswith("sweep"):   # (level 0 divides by the empty row's zero diagonal)
            assert value[lone] == alone.get(what, xh[lone]), what
        assert rel_err(value[rest], ref[what]) <= (1e-13 if precision == H.F64 else 8e-6), what
