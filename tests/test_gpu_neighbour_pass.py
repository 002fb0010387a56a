"""The neighbour pass (lists and PSE sum) where its units end: cells of 1 to 9 particles (groups of
four), 1 to 1,500 candidates (chunks of 64, the last one partial or full), rows shorter than a list,
grids whose stencil is cut off at every face.

Lists against numpy's over all pairs (the same rounding of r^2, so exact); the PSE rate against the
sum in numpy's 64 bits over the 5 x 5 x 5 cells.  Tolerances of the rate from the arithmetic: at most
1,500 terms of a few roundings each of mixed sign, 1e-12 of the largest rate (FP64); FP32 terms, a
handful of 2^-24 each, 1e-5.
"""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api

pytestmark = pytest.mark.gpu

H, MASS, RHO0, ALPHA = 7.5e-4, 5e-10, 4.43, 3e-8
# particles, edge of the box they fill in cells: from one particle to 1,500 candidates of one cell, and
# 300 particles among 216,000 cells
CLOUDS = [(1, 1.0), (2, 1.0), (3, 0.9), (5, 0.9), (9, 0.9), (63, 2.5), (64, 2.5), (65, 2.5), (127, 3.0), (128, 3.0),
          (129, 4.5), (700, 4.5), (833, 4.9), (1500, 4.9), (400, 11.0), (300, 60.0)]


def setup(n, box, precision, cap, heat):
    rng = np.random.default_rng(n)
    api.reset_globals()
    api.constants_reset()
    api.set_options(cspm=False, heat=heat, single_sqrt=False, max_neighbours=cap)
    ph = api.make_phys_constants()
    ph.rho0, ph.K, ph.G, ph.mass = RHO0, 1.2, 0.4, MASS
    t = api.make_trml_constants()
    t.cp, t.k, t.alpha, t.T_init = 5e-6, 7e-13, ALPHA, 300.0
    api.actions_setup_physical_constants(ph)
    api.interactions_setup_physical_constants(ph)
    api.interactions_setup_thermal_constants_workpiece(t)
    pos = rng.uniform(0.0, box * H, (n, 3))
    c = dict(pos=pos, rho=RHO0 * (1 + rng.uniform(-5e-3, 5e-3, n)), T=300 + rng.uniform(0, 400, n),
             h=H * rng.uniform(0.8, 1.0, n))
    p = api.particle_gpu(pos, None, c["rho"], c["T"], c["h"], None, None, None, precision=precision)
    # a box no wider than the cloud: the stencils of the outer cells are cut off
    g = api.grid_gpu_green(n, pos.min(0), pos.max(0), H)
    g.sort(p)
    order = p.download(_lib.F_ID).astype(int)
    return {k: v[order] for k, v in c.items()}, p, g


def cells(c, g):
    lo = np.array([g.bbmin_x(), g.bbmin_y(), g.bbmin_z()])
    return ((c["pos"] - lo) / g.dx()).astype(int)


@pytest.mark.parametrize("cap", [2048, 12])
def test_lists_match_all_pairs(hip_device, cap):
    for n, box in CLOUDS:
        c, p, g = setup(n, box, _lib.MFG_FP64, cap, _lib.MFG_HEAT_NONE)
        x = c["pos"]
        d = x[:, None] - x[None]
        r2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
        hit = (r2 >= 1e-8) & (r2 < (4 * c["h"] * c["h"])[:, None])
        want = [np.flatnonzero(hit[i]) for i in range(n)]
        most = max(len(w) for w in want)
        if most > cap:  # the rows keep the first entries and the overflow is an error
            with pytest.raises(_lib.MfgError):
                g.neighbours(p, cap)
            continue
        counts, lists = g.neighbours(p, max(most, 1))
        for i in range(n):
            assert counts[i] == len(want[i]), (n, box, i)
            np.testing.assert_array_equal(lists[i, :counts[i]], want[i], err_msg=f"{n} {box} {i}")


@pytest.mark.parametrize("precision,tol", [(_lib.MFG_FP64, 1e-12), (_lib.MFG_FP32_KAHAN, 1e-5)], ids=["fp64", "fp32"])
def test_pse_rate_matches_all_pairs(hip_device, precision, tol):
    for n, box in CLOUDS:
        c, p, g = setup(n, box, precision, 2048, _lib.MFG_HEAT_PSE)
        api.interactions_heat_pse(p, g)
        got = p.download(_lib.F_T_T)
        cell, x, h = cells(c, g), c["pos"], c["h"][:, None]
        near = (np.abs(cell[:, None] - cell[None]) <= 2).all(-1)
        r2 = ((x[:, None] - x[None]) ** 2).sum(-1)
        w = 4 / (h ** 5 * np.pi * np.sqrt(np.pi)) * np.exp(-r2 / (h * h)) * near
        want = ALPHA * (w * (c["T"][None] - c["T"][:, None]) * (MASS / c["rho"])[None]).sum(1)
        scale = np.abs(want).max()
        err = np.abs(got - want).max() / scale if scale > 0 else np.abs(got).max()
        assert err <= tol, (n, box, err)
