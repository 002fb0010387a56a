"""Sets beyond 32-bit offsets and launches: FP64 records of 192 bytes pass 4 GiB at 22.4M particles, FP32 records of
112 at 38.3M, the neighbour pass's candidates of 32 bytes at 134.2M; a wavefront for each of 67.1M occupied cells
passes the 2^32 threads of a launch.

A cubic lattice of spacing 1 with a support between 1 and sqrt(2): every particle has its up to six lattice
neighbours, visited in the same order everywhere, and the velocity field v = L x of constant L does not depend on
x.  So after one step all inner x-planes have the same rate of density, to the bit, in every precision: one
that came from records elsewhere in the array differs.  In FP64 the corrected gradient also gives the exact
rho_t = -rho tr(L) at every particle, on the faces too: six terms of a few roundings each on coordinates of up
to 290, 1e-10.
"""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api

pytestmark = pytest.mark.gpu

TRACE = -2e-3 + 3e-3


def lattice(n1, precision, locked=True):
    n, h = n1 ** 3, 0.675
    pos = np.zeros((n1, n1, n1, 4))
    for k in range(3):
        pos[..., k] = np.arange(n1, dtype=float).reshape([-1 if a == k else 1 for a in range(3)])
    pos = pos.reshape(n, 4)
    vel = pos * [0.0, -2e-3, 3e-3, 0.0]
    api.reset_globals()
    api.constants_reset()
    api.set_options(cspm=True, heat=_lib.MFG_HEAT_NONE, single_sqrt=False, max_neighbours=8)
    phys = api.make_phys_constants()
    phys.rho0 = phys.K = phys.G = phys.mass = 1.0
    corr = api.make_corr_constants()
    corr.alpha = corr.beta = 1.0
    corr.eta = 0.1
    api.actions_setup_physical_constants(phys)
    api.interactions_setup_physical_constants(phys)
    api.interactions_setup_corrector_constants(corr)
    api.global_time_dt = api.global_time_current = 1e-6
    one = np.ones(n)
    p = api.particle_gpu(pos, vel, one, one, h * one, None, None, None, precision=precision)
    g = api.grid_gpu_green(n, np.full(3, -0.5), np.full(3, n1 - 0.5), h) if locked else api.grid_gpu_green(6 * n, n)
    return p, g


def check_planes(p, n1):
    rho_t = np.empty(n1 ** 3)
    rho_t[p.download(_lib.F_ID).astype(np.int64)] = p.download(_lib.F_RHO_T)
    planes = rho_t.reshape(n1, -1)
    bad = np.flatnonzero((planes[1:-1] != planes[1]).any(1)) + 1
    assert len(bad) == 0, (len(bad), bad[:3])
    # in FP32 the planes are to be right, not only alike
    assert np.abs(rho_t / -TRACE - 1.0).max() <= (1e-10 if p.precision == _lib.MFG_FP64 else 1e-2)


@pytest.mark.parametrize("form", ["step", "unlocked", "batch"])
@pytest.mark.parametrize("precision,n1", [(_lib.MFG_FP64, 290), (_lib.MFG_FP32_KAHAN, 344), (_lib.MFG_FP32_WIDE, 344)],
                         ids=["fp64", "kahan", "wide"])
def test_records_beyond_4_gib(hip_device, precision, n1, form):
    if form == "unlocked" and precision != _lib.MFG_FP64:
        pytest.skip("the FP32 kernels are the same on either grid")
    p, g = lattice(n1, precision, locked=form != "unlocked")
    if form == "batch":
        b = api.batch()
        b.add(p, g)
        b.step()
    else:
        api.leap_frog(p.N_init, g.num_cell()).step(p, g)
    check_planes(p, n1)


@pytest.mark.parametrize("n1,form", [(409, "step"), (409, "batch"), (513, "step"), (513, "batch")])
def test_more_cells_than_a_launch_holds(hip_device, n1, form):
    """68.4M particles (409 a side) in 3.3 cells each, and 135M, whose candidates are beyond 4 GiB."""
    p, g = lattice(n1, _lib.MFG_FP32_KAHAN)
    api.pair_stats_enable(form == "step")
    try:
        if form == "batch":
            b = api.batch()
            b.add(p, g)
            b.step()
        else:
            api.leap_frog(p.N_init, g.num_cell()).step(p, g)
            assert p.pair_stats()[1] == 6 * n1 ** 2 * (n1 - 1)
        check_planes(p, n1)
    finally:
        api.pair_stats_enable(False)
