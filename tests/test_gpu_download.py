"""Fields of every particle to host memory at both sides of the staged size (4 MB: 58,254 symmetric
tensors, 174,762 vectors, 524,288 scalars): what was uploaded comes back, element for element.  Copies
only, so exact; flags come back as the value class they were set to."""
import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api

pytestmark = pytest.mark.gpu

F64 = {1: ("F_H", "F_RHO", "F_EPS_PL", "F_EPS_PL_DOT", "F_T", "F_RHO_T", "F_T_T"),
       3: ("F_POS", "F_VEL", "F_VEL_BC", "F_FC", "F_FT", "F_POS_T", "F_VEL_T"), 9: ("F_S", "F_S_T")}


@pytest.mark.parametrize("n", [1, 3, 255, 257, 14563, 58254, 58255, 174762, 174763, 524288, 524289])
def test_fields_come_back(hip_device, n):
    rng = np.random.default_rng(n)
    api.reset_globals()
    p = api.particle_gpu(rng.normal(size=(n, 3)), None, np.ones(n), np.ones(n), np.ones(n), None, None, None)
    for turn in range(2):  # the second finds the staging buffer as the first left it
        sent = {}
        for w, names in F64.items():
            for name in names:
                v = rng.normal(size=(n, w))
                if w == 9:
                    m = v.reshape(n, 3, 3)
                    v = (m + m.transpose(0, 2, 1)).reshape(n, 9)
                v = v[:, 0] if w == 1 else v
                sent[name] = v
        sent["F_FIXED"] = rng.integers(0, 3, n).astype(float)
        sent["F_TOOL"] = rng.integers(0, 3, n).astype(float)
        sent["F_BLANKED"] = rng.integers(0, 2, n).astype(float)
        for name, v in sent.items():
            p.upload(getattr(_lib, name), v)
        for name, v in sent.items():
            got = p.download(getattr(_lib, name))
            assert np.array_equal(got.reshape(v.shape), v), (name, turn)
        assert np.array_equal(p.download(_lib.F_ID), np.arange(n))
