"""The counting sort at the edges of its tiles and launches: one particle to many in a cell, sets
below and above a workgroup, up to and beyond 128k cells (one scan launch or two) and 128k particles
(the order inside the cells found by the permutation or in a launch of its own), with blanked
particles, twice on the same grid and then by a step.

Against numpy's stable sort of the keys (the same divisions): whole numbers, so exact."""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api

pytestmark = pytest.mark.gpu

H = 1e-3


def expected(pos, blanked, g):
    lo = np.array([g.bbmin_x(), g.bbmin_y(), g.bbmin_z()])
    i = ((pos - lo) / g.dx()).astype(np.int64)
    key = (i[:, 0] * g.ny() + i[:, 1]) * g.nz() + i[:, 2]
    key[blanked != 0] = 2**31 - 1
    return np.argsort(key, kind="stable"), key


@pytest.mark.parametrize("n,edge", [(1, 1), (63, 1), (64, 2), (65, 2), (300, 1), (256, 15), (257, 16), (4097, 15),
                                    (5000, 52), (140000, 40), (140000, 60)])
def test_sort_is_stable(hip_device, n, edge):
    rng = np.random.default_rng(n + edge)
    api.reset_globals()
    api.constants_reset()
    api.set_options(cspm=True, heat=_lib.MFG_HEAT_NONE, single_sqrt=False, max_neighbours=512)
    ph = api.make_phys_constants()
    ph.rho0, ph.K, ph.G, ph.mass = 4.43, 1.2, 0.4, 5e-10
    api.actions_setup_physical_constants(ph)
    api.interactions_setup_physical_constants(ph)
    pos = rng.uniform(0.0, edge * H, (n, 3))
    p = api.particle_gpu(pos, None, np.full(n, 4.43), np.full(n, 300.0), np.full(n, H), None, None, None)
    g = api.grid_gpu_green(n, pos.min(0), np.full(3, edge * H), H)
    ids = np.arange(n)
    lf = api.leap_frog(n, g.num_cell())
    api.global_time_dt = 1e-15
    for turn in range(3):
        pos = np.maximum(rng.uniform(0.0, edge * H, (n, 3)), pos.min(0))
        blanked = (rng.random(n) < 0.1).astype(float) if n > 1 else np.zeros(n)
        p.upload(_lib.F_POS, pos)
        p.upload(_lib.F_BLANKED, blanked)
        order, key = expected(pos, blanked, g)
        if turn < 2:
            g.sort(p)
        else:
            lf.step(p, g)
        ids = ids[order]
        assert np.array_equal(p.download(_lib.F_IDX), order), turn
        assert np.array_equal(p.download(_lib.F_HASH), key[order]), turn
        assert np.array_equal(p.download(_lib.F_ID), ids), turn
