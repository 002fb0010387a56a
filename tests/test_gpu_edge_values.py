"""Particles whose own values lie outside the ordinary range, one step against the oracle: which particles of their
neighbourhood the NaN/Inf guard (src/actions_gpu.cu:302-331) blanks, exactly, and the rates of the others there.

- A negative density has no sound speed (NaN).  The viscosity takes it only where a pair approaches
  (src/interactions_gpu.cu:411-423), so the neighbours that recede keep finite rates.
- A smoothing length of zero has an empty list and an infinite kernel; without neighbours every sum is zero.
- A NaN smoothing length excludes no candidate (src/kernels.cuh:41), so the particle's rates are NaN; its
  neighbours take it into their viscosity alone.

Tolerances from the arithmetic: FP64 sums of about 100 terms of a few roundings each, 1e-11 of a field's norm;
FP32 terms, 2^-24 each with a handful of operations and cancellation of the stress sum by up to ten, 1e-4.
"""
import numpy as np
import pytest

import helpers
import oracle as O
from iwf_mfree_gpu_3d_amd import _lib, api, scenes
from test_gpu_parity import perturbed_scene, rel_err

pytestmark = pytest.mark.gpu


def spoil(sc, what):
    """The particles nearest to three points of the workpiece, spoiled; their indices."""
    wp = np.flatnonzero(sc.tool_p == 0)
    lo, hi = sc.pos[wp].min(0), sc.pos[wp].max(0)
    at = [lo + f * (hi - lo) for f in (0.2, 0.5, 0.8)]
    ks = [int(wp[np.argmin(np.linalg.norm(sc.pos[wp] - a, axis=1))]) for a in at]
    if what == "negative density":
        sc.rho[ks] *= -0.3
    elif what == "no smoothing length":
        sc.h[ks] = 0.0
    elif what == "NaN smoothing length":
        sc.h[ks] = np.nan
    return ks


@pytest.mark.parametrize("what", ["negative density", "no smoothing length", "NaN smoothing length"])
@pytest.mark.parametrize("scale", [0.5, 1.0])  # about 1,000 and 8,000 particles: either lane count of the pair pass
@pytest.mark.parametrize("precision,locked,tol", [(_lib.MFG_FP64, True, 1e-11), (_lib.MFG_FP64, False, 1e-11),
                                                  (_lib.MFG_FP32_KAHAN, True, 1e-4), (_lib.MFG_FP32_WIDE, True, 1e-4)],
                         ids=["fp64", "fp64_unlocked", "kahan", "wide"])
def test_guard_blanks_what_the_oracle_blanks(hip_device, precision, locked, tol, scale, what):
    sc = perturbed_scene(1, scale, 7)
    ks = spoil(sc, what)
    sim = helpers.oracle_from_scene(sc)
    dt = sc.params.dt
    sim.set_time(dt, dt)
    parts, grid = scenes.setup_cut(sc, precision=precision, max_neighbours=1024)  # a whole stencil
    if not locked:
        grid = api.grid_gpu_green(4 * grid.num_cell() + 1000, sc.n)
    api.global_time_current = dt
    assert sim.run(1) == 0
    scenes.run(api.leap_frog(sc.n, grid.num_cell()), parts, grid, 1)
    og = np.argsort(parts.download(_lib.F_ID).astype(np.int64))
    oo = np.argsort(sim.field(O.F_ID).astype(np.int64))
    blanked = sim.field(O.F_BLANKED)[oo]
    # inside the support, where pairs interact (the oracle also adds 0 * NaN for the rest of the stencil)
    near = np.min([np.linalg.norm(sc.pos - sc.pos[k], axis=1) for k in ks], axis=0) < 1.99 * sc.params.h
    np.testing.assert_array_equal(parts.download(_lib.F_BLANKED)[og][near], blanked[near])
    keep = (blanked != 1.0) & near
    if what != "no smoothing length":
        assert blanked[ks].all() and keep.sum() > 20, "the particles are blanked, neighbours that recede are not"
    else:
        assert keep[ks].all()
    for f, of in [(_lib.F_POS_T, O.F_POS_T), (_lib.F_VEL_T, O.F_VEL_T), (_lib.F_RHO_T, O.F_RHO_T)]:
        g, o = parts.download(f)[og][keep], sim.field(of)[oo][keep]
        assert np.isfinite(g).all()
        assert rel_err(g, o) < tol, (f, rel_err(g, o))


@pytest.mark.parametrize("precision", [_lib.MFG_FP64, _lib.MFG_FP32_KAHAN], ids=["fp64", "fp32"])
def test_infinite_temperature_heats_to_infinity(hip_device, precision):
    """The PSE rate of a particle beside one of infinite temperature is infinite, not NaN (a chunk of candidates has
    unused lanes, which are to add nothing)."""
    h, n = 7.5e-4, 70
    rng = np.random.default_rng(5)
    api.reset_globals()
    api.constants_reset()
    api.set_options(cspm=False, heat=_lib.MFG_HEAT_PSE, single_sqrt=False)
    phys = api.make_phys_constants()
    phys.rho0, phys.K, phys.G, phys.mass = 4.43, 1.2, 0.4, 5e-10
    trml = api.make_trml_constants()
    trml.cp, trml.k, trml.alpha, trml.T_init = 5e-6, 7e-13, 3e-8, 300.0
    api.actions_setup_physical_constants(phys)
    api.interactions_setup_physical_constants(phys)
    api.interactions_setup_thermal_constants_workpiece(trml)
    pos = rng.uniform(0.0, h, (n, 3))  # one cell's stencil
    T = np.full(n, 300.0)
    T[0] = np.inf
    p = api.particle_gpu(pos, None, np.full(n, 4.43), T, np.full(n, h), None, None, None, precision=precision)
    g = api.grid_gpu_green(n, pos.min(0), pos.max(0), h)
    g.sort(p)
    hot = p.download(_lib.F_ID) == 0
    api.interactions_heat_pse(p, g)
    rate = p.download(_lib.F_T_T)
    assert np.isnan(rate[hot]).all() and (rate[~hot] == np.inf).all()
