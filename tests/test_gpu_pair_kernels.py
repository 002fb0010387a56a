"""The two FP64 pair kernels against each other with every term at work: the one-walk sums (4 and 16 lanes a
particle, locked grid) and the sums in the reference's order (one lane, unlocked grid) of the same particles.

A cut with pressure of both signs, deviatoric and artificial stress, viscosity, XSPH and Brookshaw heat.  The
kernels round differently everywhere.  Tolerance from the arithmetic: sums of about 100 terms of ten roundings
each, cancelling by up to ten, the fourth power of the artificial stress four times that: 100 * 10 * 1.1e-16 *
10 * 4 = 4.4e-12, so 1e-11 of a field's largest value.
"""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api, scenes
from test_gpu_parity import perturbed_scene

pytestmark = pytest.mark.gpu

RATES = [_lib.F_V_DER, _lib.F_S_DER, _lib.F_VEL_T, _lib.F_POS_T, _lib.F_T_T]


def rates(sc, S, locked):
    parts, grid = scenes.setup_cut(sc)
    if not locked:
        grid = api.grid_gpu_green(4 * grid.num_cell() + 1000, sc.n)
        grid.update_geometry(parts)
    parts.upload(_lib.F_S, S)
    grid.sort(parts)
    api.material_eos(parts)
    api.corrector_artificial_stress(parts)
    api.interactions_monaghan(parts, grid)
    place = np.argsort(parts.download(_lib.F_ID).astype(np.int64))
    return [parts.download(f)[place] for f in [*RATES, _lib.F_R]]


@pytest.mark.parametrize("scale", [0.5, 1.0])  # 1,000 particles: 16 lanes; 8,000: 4
def test_one_walk_matches_the_ordered_sums(hip_device, scale):
    sc = perturbed_scene(1, scale, 11)
    rng = np.random.default_rng(3)
    sc.rho *= 1.0 + rng.uniform(-5e-3, 5e-3, sc.n)
    sc.T += rng.uniform(0.0, 300.0, sc.n)
    s = rng.uniform(-5e-3, 5e-3, (sc.n, 6))
    a, b = rates(sc, s[:, [0, 3, 5, 3, 1, 4, 5, 4, 2]], True), rates(sc, s[:, [0, 3, 5, 3, 1, 4, 5, 4, 2]], False)
    assert np.count_nonzero(np.abs(a[-1]).max(1)) > sc.n // 10, "artificial stress is at work"
    for f, x, y in zip([*RATES, _lib.F_R], a, b):
        scale_f = np.abs(y).max()
        assert scale_f > 0, f
        assert np.abs(x - y).max() <= 1e-11 * scale_f, (f, np.abs(x - y).max() / scale_f)
    assert any((x != y).any() for x, y in zip(a[:2], b[:2])), "two kernels, not one"
