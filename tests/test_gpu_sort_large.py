"""The counting sort where its prefix sums go in two levels: from 16,384 workgroups of 256 particles (4.2M) and
16,384 tiles of 4,096 cells (67M) on, either, both or neither, with every tenth particle blanked at random.  Keys,
permutation and tables are whole numbers: equal to numpy's stable sort."""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api

pytestmark = pytest.mark.gpu

FEW, MANY = 300_000, 4_194_304 + 70_001  # particles; MANY: 273 workgroups more than 16,384
SMALL, LARGE = (90, 70, 110), (420, 401, 407)  # cells: 693,000 and 68.5M (16,735 tiles)


def particles(n, cells, h):
    rng = np.random.default_rng(n)
    cell = np.stack([rng.integers(0, c, n) for c in cells], axis=1)
    api.reset_globals()
    api.constants_reset()
    api.set_options(cspm=False, heat=_lib.MFG_HEAT_NONE, single_sqrt=False, max_neighbours=8)
    one = np.ones(n)
    # supports smaller than a cell: no neighbours
    p = api.particle_gpu((cell + 0.5) * h, None, one, one, 0.3 * h * one, None, None, None)
    blanked = rng.random(n) < 0.1
    p.upload(_lib.F_BLANKED, blanked.astype(float))
    key = (cell[:, 0] * cells[1] + cell[:, 1]) * cells[2] + cell[:, 2]
    return p, np.where(blanked, 2 ** 31 - 1, key)


@pytest.mark.parametrize("form", ["sort", "step", "batch"])
@pytest.mark.parametrize("n,cells", [(FEW, SMALL), (MANY, SMALL), (FEW, LARGE), (MANY, LARGE)],
                         ids=["neither", "particles", "cells", "both"])
def test_sort_matches_numpy(hip_device, n, cells, form):
    h = 0.5
    p, key = particles(n, cells, h)
    # the box of a grid is widened by 1e-6 on either side: a little narrower here, for as many cells as said
    g = api.grid_gpu_green(n, np.zeros(3), np.array(cells) * h - 1e-3, h)
    assert g.num_cell() == np.prod(cells)
    g.set_hard_blank(True)
    api.global_time_dt = api.global_time_current = 1e-6
    if form == "sort":
        g.sort(p)
    elif form == "step":
        api.leap_frog(n, g.num_cell()).step(p, g)
    else:
        b = api.batch()
        b.add(p, g)
        b.step()
    order = np.argsort(key, kind="stable")
    np.testing.assert_array_equal(p.download(_lib.F_ID).astype(np.int64), order)
    np.testing.assert_array_equal(p.download(_lib.F_HASH).astype(np.int64), key[order])
    assert p.N == int((key < 2 ** 31 - 1).sum())
