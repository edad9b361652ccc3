"""Launch schedules where they are used: one right-hand side on levels from 5 up (levels 1 to 4 run apply, residual and
sweeps without one).  Every schedule computes the same values in the same order, bit for bit."""
import numpy as np
import pytest

from helpers import rel_err, say

pytestmark = pytest.mark.gpu

# (rows, waves, block, kind): row windows, flat slab windows, LDS slab tiles, columns
SCHEDULES = [(1, 1, 1, 0), (3, 2, 2, 0), (4, 4, 8, 0), (8, 4, 4, 0), (64, 2, 8, 0), (2, 1, 8, 0), (13, 4, 2, 0), (7, 1, 4, 0),
             (1, 1, 1, 1), (4, 2, 2, 1), (8, 4, 4, 1), (3, 1, 8, 1), (2, 2, 1, 1), (64, 4, 4, 1),
             (4, 4, 1, 2), (3, 4, 2, 2), (8, 2, 5, 2), (12, 4, 64, 2), (2, 1, 3, 2),
             (1, 1, 1, 3), (2, 2, 2, 3), (3, 4, 4, 3), (5, 1, 2, 3), (16, 2, 2, 3), (64, 4, 1, 3), (4, 8, 9, 3), (16, 16, 1, 3),
             (2, 16, 10, 3)]


@pytest.mark.parametrize("level", [5, 6])
@pytest.mark.parametrize("precision", [0, 1])
def test_every_kind_bitwise(level, precision, gpu_ctx):
    import hyteg_amd as H
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), 1, 1, 1), gpu_ctx)
    rng = np.random.default_rng(level)
    xh, bh, yh = rng.standard_normal((3, S.owned_count(level)))
    A = H.P1ConstantLaplaceOperator(S, level, level)
    x, b, y = (H.P1Function(k, S, level, level, precision=precision) for k in "xby")
    b.upload(level, bh)
    S.set_cell_sor(level, 0)    # (level 5 sweeps a cell per workgroup, level 6 by colour passes on the schedule)

    def run():
        out = []
        x.upload(level, xh)
        y.upload(level, yh)
        A.apply(x, y, level, H.INNER)
        out.append(y.download(level))
        y.upload(level, yh)
        A.apply(x, y, level, H.INNER, H.ADD)
        out.append(y.download(level))
        A.residual(x, b, y, level, H.INNER)
        out.append(y.download(level))
        A.smooth_sor(x, b, 0.8, level, H.INNER)
        A.smooth_sor_backwards(x, b, 0.8, level, H.INNER)
        out.append(x.download(level))
        return out

    S.set_schedule(level)
    ref, ran = run(), {}
    for rows, waves, block, kind in SCHEDULES:
        try:
            S.set_schedule(level, rows, waves, block, kind)
        except H._lib.HymiError:    # a band too large for LDS
            assert kind == 2
            continue
        say(f"[schedules] level {level} precision {precision}: kind {kind} rows {rows} waves {waves} block {block}")
        ran[kind] = ran.get(kind, 0) + 1
        for got, want in zip(run(), ref):
            assert np.array_equal(got, want), (rows, waves, block, kind)
    S.set_schedule(level)
    assert set(ran) == {0, 1, 2, 3}


@pytest.mark.parametrize("level", [5, 6])
def test_graph_recaptured_after_schedule_change(level, gpu_ctx):
    """The captured cycle's residual on this level reads the schedule's work units, which a new schedule frees; the epoch
    that makes the next replay capture again is checked on the host (test_schedule_epoch.py)."""
    import hyteg_amd as H
    say(f"[graph schedule] level {level}")
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), 2, 2, 2), gpu_ctx)
    A = H.P1ConstantLaplaceOperator(S, 0, level)
    b, x, x2 = (H.P1Function(k, S, 0, level) for k in ("b", "x", "x2"))
    b.interpolate_modes(np.array([[1.0, 1, 1, 1], [0.3, 3, 5, 2]]), level)
    gmg = H.GeometricMultigridSolver(S, H.SORSmoother(1.0), H.CGSolver(S, 0, 0), H.P1toP1LinearRestriction(),
                                     H.P1toP1LinearProlongation(), 0, level, 2, 2)
    for schedule in ((), (2, 4, 2, 3), (4, 2, 1, 1), (16, 4, 1, 3)):
        S.set_schedule(level, *schedule)
        for _ in range(2):
            gmg.solve(A, x, b, level)
            gmg.solve_graph(A, x2, b, level, 1)
            _ = x.dotGlobal(x, level, H.INNER)      # eager work and a wait between the replays
            assert rel_err(x2.download(level), x.download(level)) == 0.0, schedule
    S.set_schedule(level)


def _difference(H, S, a, b, level, precision):
    d = H.P1Function("d", S, level, level, precision=precision)
    d.assign([1.0, -1.0], [a, b], level, H.ALL)
    return d.dotGlobal(d, level, H.ALL)


@pytest.mark.parametrize("n,level", [(1, 1), (2, 2), (1, 4), (2, 5), (1, 6), (2, 8)])
@pytest.mark.parametrize("precision", [0, 1])
def test_prolongation_replaces(n, level, precision, gpu_ctx):
    """Prolongation with Replace gives the bits of adding to zeroed points, and leaves alone what the flag leaves out.
    48 macro-tets at level 8 are 0.54 and 1.1 GB: the branch that streams past the memory-side cache."""
    import hyteg_amd as H
    say(f"[prolongation] n={n} level={level} precision={precision}")
    S = H.PrimitiveStorage(H.MeshInfo.meshCuboid((0, 0, 0), (1, 1, 1), n, n, n), gpu_ctx)
    a, b = (H.P1Function(k, S, level - 1, level, precision=precision) for k in "ab")
    coarse = np.array([[1.0, 1.5, 2.5, 0.5], [0.7, 3.5, 1.5, 4.5]])
    fine = np.array([[0.9, 2.5, 0.5, 1.5]])
    transfer = H.P1toP1LinearProlongation()
    for flag in (H.INNER, H.ALL):
        for f in (a, b):
            f.interpolate_modes(coarse, level - 1)
            f.interpolate_modes(fine, level)
        transfer.prolongate(a, level - 1, flag)
        b.interpolate(0.0, level, flag)
        transfer.prolongateAndAdd(b, level - 1, flag)
        assert a.dotGlobal(a, level, H.ALL) > 0.0
        assert _difference(H, S, a, b, level, precision) == 0.0, flag
        if flag == H.INNER:     # the boundary keeps the fine values
            b.interpolate_modes(fine, level)
            b.interpolate(0.0, level, H.INNER), a.interpolate(0.0, level, H.INNER)
            assert b.dotGlobal(b, level, H.ALL) > 0.0
            assert _difference(H, S, a, b, level, precision) == 0.0
