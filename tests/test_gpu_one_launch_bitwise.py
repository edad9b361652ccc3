"""The one-launch apply, residual, sweeps and the owner-table restriction of small levels against the separate launches, bit
for bit.  A node that no tetrahedron uses, appended to the mesh, sends the same calls the separate way and changes
nothing else.  Sweeps one by one (a copy follows each) and, through cycles of 2 and 3 smoothing steps, in sequences; the
cycles to 64 eps, since the sums over the vertices in the coarsest level's CG have one more term.  After the sweeps the
cells' micro-vertices (the closure copies included) equal too."""
import numpy as np
import pytest

from helpers import MESHES, read_gmsh, rel_err, say

pytestmark = pytest.mark.gpu


def _mesh(kind):
    if kind == "cube":
        g = np.arange(3) / 2.0
        X = np.array([[x, y, z] for z in g for y in g for x in g])
        corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
        split = ((4, 5, 7, 3), (0, 3, 1, 4), (4, 1, 5, 3), (5, 6, 7, 2), (1, 3, 2, 5), (7, 2, 3, 5))
        C = [[(i + corner[k][0]) + 3 * (j + corner[k][1]) + 9 * (m + corner[k][2]) for k in tet]
             for i in range(2) for j in range(2) for m in range(2) for tet in split]
        return X, np.array(C, dtype=np.int32)
    return read_gmsh(f"{MESHES}/{kind}")


@pytest.mark.parametrize("kind", ["cube", "regular_octahedron_8el.msh", "pyramid_2el.msh"])
@pytest.mark.parametrize("level", [1, 2, 3, 4])
@pytest.mark.parametrize("precision", [0, 1])
def test_same_bits(kind, level, precision, gpu_ctx):
    import hyteg_amd as H
    say(f"[one launch] {kind} level={level} precision={precision}")
    X, C = _mesh(kind)

    def results(X, extra):
        S = H.PrimitiveStorage(H.MeshInfo.fromArrays(X, C), gpu_ctx)
        keep = np.arange(S.owned_count(level)) != (len(X) - 1 if extra else -1)
        keep_c = np.arange(S.owned_count(level - 1)) != (len(X) - 1 if extra else -1)
        xh, bh, yh = (np.zeros(len(keep)) for _ in range(3))
        for k, h in enumerate((xh, bh, yh)):
            h[keep] = np.random.default_rng([level, k]).standard_normal(keep.sum())
        A = H.P1ConstantLaplaceOperator(S, 0, level)
        x, b, y = (H.P1Function(k, S, 0, level, precision=precision) for k in "xby")
        x.upload(level, xh), b.upload(level, bh)
        out = {}
        for flag in (H.INNER, H.ALL):
            for what in ("replace", "add", "residual"):
                y.upload(level, yh)
                if what == "residual":
                    A.residual(x, b, y, level, flag)
                else:
                    A.apply(x, y, level, flag, H.ADD if what == "add" else H.REPLACE)
                out[what, flag] = y.download(level)[keep]
            H.P1toP1LinearRestriction().restrict(y, level, flag)
            out["restrict", flag] = y.download(level - 1)[keep_c]
            for k in range(2):
                A.smooth_sor(x, b, 0.9, level, flag)
                out["sweep", k, flag] = x.download(level)[keep]
                out["micro-vertices", k, flag] = x.download_micro_vertices(level)
        for steps in (2, 3):
            gmg = H.GeometricMultigridSolver(S, H.SORSmoother(0.9), H.CGSolver(S, 0, 0), H.P1toP1LinearRestriction(),
                                             H.P1toP1LinearProlongation(), 0, level, steps, steps)
            b.interpolate(0.0, level), b.interpolate(1.0, level, H.INNER)
            if extra:
                bh = b.download(level)
                bh[~keep] = 0.0
                b.upload(level, bh)
            gmg.solve(A, x, b, level)
            out["cycle", steps] = x.download(level)[keep]
        return out

    one, separate = results(X, False), results(np.vstack([X, [[9.0, 9.0, 9.0]]]), True)
    for what in one:
        if what[0] == "cycle":
            assert rel_err(one[what], separate[what]) <= 64 * np.finfo(("f8", "f4")[precision]).eps, what
        else:
            assert np.array_equal(one[what], separate[what]), what
