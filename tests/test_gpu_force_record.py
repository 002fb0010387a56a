"""The recorded tool force against the contact forces of the particles it sums, at sets of 2, 32, 250
and 550 workgroups (the sum takes 256 at a time).

The record is a float sum: within a workgroup by halves (8 additions deep) and then workgroup by
workgroup, so its error is at most (8 + 550) 2^-24, 3.3e-5, of the sum of the magnitudes."""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [4, 10, 20, 26])
def test_record_is_the_sum(hip_device, nz):
    sc = scenes.Scene(1, 1.0, 1, nx=4 * nz, ny=2 * nz, nz=nz)
    p, g = scenes.setup_cut(sc)
    lf = api.leap_frog(sc.n, g.num_cell())
    api.global_time_current = sc.params.dt
    scenes.run(lf, p, g, 39)
    scenes.run(lf, p, g, 1, record_forces=True)
    f = (p.download(_lib.F_FC) + p.download(_lib.F_FT))[: p.N]
    got = api.global_tool_forces.get_forces_host().reshape(-1, 3)[0]
    assert np.abs(f).max() > 0, "the tool must be in contact"
    assert np.abs(got - f.sum(0)).max() <= (8 + 550) * 2.0**-24 * np.abs(f).sum(0).max()
