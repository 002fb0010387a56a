"""Fields that are made on request: an error of the queued steps comes before the missing array and, once the array
is there, instead of its values."""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api, scenes

pytestmark = pytest.mark.gpu

ON_REQUEST = [_lib.F_V_DER, _lib.F_S_DER, _lib.F_N, _lib.F_P, _lib.F_R]


def code_of(parts, field):
    with pytest.raises(_lib.MfgError) as e:
        parts.download(field)
    return e.value.code


@pytest.mark.parametrize("field", ON_REQUEST)
def test_queued_errors_come_first(hip_device, field):
    sc = scenes.Scene(1, 0.5, 3)
    parts, grid = scenes.setup_cut(sc, max_neighbours=32)  # about 100 neighbours a particle: over the capacity
    assert code_of(parts, field) == _lib.MFG_ERR_STATE
    lf = api.leap_frog(sc.n, grid.num_cell())
    api.global_time_current = sc.params.dt
    lf.step(parts, grid)
    assert code_of(parts, field) == _lib.MFG_ERR_CAPACITY
    lf.init(parts)  # makes the arrays
    assert code_of(parts, field) == _lib.MFG_ERR_CAPACITY


def test_values_once_made(hip_device):
    sc = scenes.Scene(1, 0.5, 3)
    parts, grid = scenes.setup_cut(sc)
    grid.sort(parts)
    api.material_eos(parts)
    api.interactions_monaghan(parts, grid)
    for field in ON_REQUEST:
        a = parts.download(field)
        assert a.shape[0] == sc.n and np.isfinite(a).all()
