"""The FP32 wide sums keep the bits of earlier versions: the rounding of r^2 in the CSPM terms goes by the
neighbour's place in the list (Pair32::cspm_term, x_first), which no other test can tell from a uniform one.

The fixture holds the rates that the one-lane kernel gave for the cloud below (257 particles, lists of up to 150,
tool particles among them), before a particle's sums were spread over several lanes.
"""
import os

import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api
from test_gpu_pair_sums import DX, cloud, constants

pytestmark = pytest.mark.gpu

FIXTURE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "wide_pair_sums.npz")
FIELDS = {"x_t": _lib.F_POS_T, "v_t": _lib.F_VEL_T, "v_der": _lib.F_V_DER, "S_der": _lib.F_S_DER, "T_t": _lib.F_T_T}


def rates():
    c = cloud(257, 4242, 1.0)
    constants(_lib.MFG_HEAT_BROOKSHAW, True, True, c["h"].max(), 0)
    p = api.particle_gpu(c["pos"], c["vel"], c["rho"], c["T"], c["h"], None, c["tool"], c["S9"],
                         precision=_lib.MFG_FP32_WIDE)
    g = api.grid_gpu_green(257, c["pos"].min(0) - DX, c["pos"].max(0) + DX, float(c["h"].max()))
    g.sort(p)
    api.material_eos(p)
    api.interactions_monaghan(p, g)
    return {name: p.download(f) for name, f in FIELDS.items()}


def test_wide_sums_keep_their_bits(hip_device):
    want, got = np.load(FIXTURE), rates()
    for name in FIELDS:
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)
