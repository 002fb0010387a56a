"""The first use of a grid whose memory held another grid's tables: no particle has a neighbour before a sort, and
the first sort, step or batched step is that of any other grid of the geometry, to the bit."""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api, scenes
from test_gpu_parity import perturbed_scene

pytestmark = pytest.mark.gpu

FIELDS = [_lib.F_ID, _lib.F_POS, _lib.F_VEL, _lib.F_RHO, _lib.F_S]


def first_use(form, dirty):
    sc = perturbed_scene(1, 1.0, 7)
    if dirty:  # a sorted grid of the same size, freed: its memory comes back for the next one
        parts, grid = scenes.setup_cut(sc)
        grid.sort(parts)
        api.synchronize()
        del grid
    parts, grid = scenes.setup_cut(sc)
    api.global_time_current = sc.params.dt
    if form == "unsorted":
        api.material_eos(parts)
        api.interactions_monaghan(parts, grid)
        return [parts.download(_lib.F_V_DER), parts.download(_lib.F_S_DER)]
    if form == "sort":
        grid.sort(parts)
    elif form == "step":
        api.leap_frog(sc.n, grid.num_cell()).step(parts, grid)
    elif form == "other stream":
        api.stream_pool(2)
        api.select_stream(1)
        try:
            grid.sort(parts)
            api.synchronize()
        finally:
            api.select_stream(0)
    else:
        b = api.batch()
        b.add(parts, grid, api.global_tool, api.global_blanking)
        b.step(2, use_graph=True)
    return [parts.download(f) for f in FIELDS]


@pytest.mark.parametrize("form", ["unsorted", "sort", "step", "other stream", "batch"])
def test_first_use(hip_device, form):
    clean, dirty = first_use(form, False), first_use(form, True)
    for a, b in zip(clean, dirty):
        np.testing.assert_array_equal(a, b)
    if form == "unsorted":
        assert all((a == 0.0).all() for a in dirty)
