"""Interpolation of Fourier modes at the cells' interior points by row and step factors: one mode, the most the row form
takes (8) and one more (the direct form); levels with one interior point per cell (2), one chunk of 64 points per row (5)
and two (7); half wave numbers.  Against host evaluation: the arguments reach 8.5 pi, rounded a few times, so 64 eps = 1.4e-14
per mode of amplitude 1 bounds the difference; FP32 adds its rounding of the sum."""
import numpy as np
import pytest

from helpers import mesh_pair, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [("cube", 1), ("gmsh", "regular_octahedron_8el.msh")])
@pytest.mark.parametrize("level", [2, 5, 7])
@pytest.mark.parametrize("n_modes", [1, 8, 9])
@pytest.mark.parametrize("precision", [0, 1])
def test_modes_match_host(kind, level, n_modes, precision, gpu_ctx):
    import hyteg_amd as H
    say(f"[modes rows] {kind} level={level} modes={n_modes} precision={precision}")
    _, S = mesh_pair(kind, gpu_ctx)
    rng = np.random.default_rng(n_modes)
    modes = np.concatenate([rng.uniform(-1, 1, (n_modes, 1)), rng.integers(1, 9, (n_modes, 3)) + 0.5], axis=1)
    f = H.P1Function("f", S, level, level, precision=precision)
    f.interpolate_modes(modes, level)
    X = S.owned_coords(level)
    ref = sum(a * np.prod(np.sin(np.pi * X * k), axis=1) for a, *k in modes)
    err = np.abs(f.download(level) - ref).max()
    say(f"  {err:.2e}")
    assert err <= n_modes * (1.4e-14 + (6e-8 if precision == H.F32 else 0.0))
