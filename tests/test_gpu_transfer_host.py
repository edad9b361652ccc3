"""Host transfers of owned values (hymi_function_upload_owned, _download_owned, _download_owned_column): the values of
every cell and face land at the points the owned-DoF order names, read back another way, and a round trip returns them,
exactly: levels without edge, face or cell interiors, one cell point (level 2), and more values than two staging
batches of 2^19 hold (level 6; level 4 with 32 right-hand sides)."""
import numpy as np
import pytest

from helpers import mesh_pair, say

pytestmark = pytest.mark.gpu


def _interior(w, dims):
    """Positions of the interior points in a primitive's index order (x fastest), for a cell (3) or a face (2)."""
    if dims == 2:
        pts = [(x, y) for y in range(w) for x in range(w - y)]
        return [k for k, (x, y) in enumerate(pts) if x >= 1 and y >= 1 and x + y <= w - 2]
    pts = [(x, y, z) for z in range(w) for y in range(w - z) for x in range(w - z - y)]
    return [k for k, (x, y, z) in enumerate(pts) if min(x, y, z) >= 1 and x + y + z <= w - 2]


@pytest.mark.parametrize("kind", [("cube", 2), ("gmsh", "pyramid_2el.msh")])
@pytest.mark.parametrize("level,nrhs", [(0, 1), (1, 1), (2, 1), (3, 1), (6, 1), (1, 32), (4, 32)])
@pytest.mark.parametrize("precision", [0, 1])
def test_owned_values_reach_their_points(kind, level, nrhs, precision, gpu_ctx):
    import hyteg_amd as H
    say(f"[owned transfer] {kind} level={level} nrhs={nrhs} precision={precision}")
    _, S = mesh_pair(kind, gpu_ctx)
    n, w = S.owned_count(level), 2 ** level + 1
    v = np.random.default_rng(level).standard_normal((n, nrhs))
    stored = v if precision == H.F64 else v.astype(np.float32).astype(np.float64)
    f = H.P1Function("f", S, level, level, precision=precision, nrhs=nrhs)
    f.upload(level, v[:, 0] if nrhs == 1 else v)
    assert np.array_equal(f.download(level).reshape(n, nrhs), stored)
    for col in {0, nrhs - 1}:
        assert np.array_equal(f.download_column(level, col), stored[:, col])
    nV, nE, nF, nC = S.counts()
    faces = nV + nE * max(0, w - 2)
    cells = n - nC * len(_interior(w, 3))
    for cls, at, dims, count in ((H.FACE, faces, 2, nF), (H.CELL, cells, 3, nC)):
        inner = _interior(w, dims)
        got = f.download_micro_vertices(level, cls).reshape(count, -1, nrhs)[:, inner]
        assert np.array_equal(got, stored[at:at + count * len(inner)].reshape(count, len(inner), nrhs))
