"""Interpolation of Fourier modes as short as the mesh resolves (wave numbers up to two fifths of the points along an edge).
A value is the sum of a sin(k pi x) sin(l pi y) sin(m pi z) with every argument rounded as written here (the factor k pi,
then its product with the coordinate): the sines of a form by row and step factors may not lose that argument's roundings,
40 eps at k = 51.  Per mode of amplitude 1: three sines of at most 4 roundings of 2^-53 each in the library and one
here, the product's two on either side and the sum's: 2e-15.  FP32 adds the rounding of the sum, 2^-24 per mode.  The
points of the cube's mesh lie on multiples of 2^-level, and so do the octahedron's, up to its corner factor."""
import numpy as np
import pytest

from helpers import mesh_pair, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [("cube", 1), ("gmsh", "regular_octahedron_8el.msh")])
@pytest.mark.parametrize("level", [2, 3, 4, 5, 7])
@pytest.mark.parametrize("n_modes", [1, 8, 9, 20])
@pytest.mark.parametrize("precision", [0, 1])
def test_short_waves_match_host(kind, level, n_modes, precision, gpu_ctx):
    import hyteg_amd as H
    _, S = mesh_pair(kind, gpu_ctx)
    rng = np.random.default_rng(n_modes + level)
    k_max = max(2, 2 * 2 ** level // 5)
    modes = np.concatenate([rng.uniform(0.5, 1, (n_modes, 1)), rng.integers(k_max // 2, k_max + 1, (n_modes, 3))], axis=1)
    f = H.P1Function("f", S, level, level, precision=precision)
    f.interpolate_modes(modes, level)
    X = S.owned_coords(level)
    ref = sum(a * np.prod(np.sin((k * np.pi)[None, :] * X), axis=1) for a, k in zip(modes[:, 0], modes[:, 1:]))
    err = np.abs(f.download(level) - ref).max()
    say(f"[modes accuracy] {kind} level={level} modes={n_modes} precision={precision}: {err:.2e}")
    assert err <= n_modes * (2e-15 + (6e-8 if precision == H.F32 else 0.0))
