"""A thread that reads a field of a set while another steps it: the reads see some step's values, and the steps
are those of a set that nobody reads, to the bit.  Fields on both sides of the download's chunk."""
import threading

import numpy as np
import pytest

from iwf_mfree_gpu_3d_amd import _lib, api, scenes
from test_gpu_parity import perturbed_scene

pytestmark = pytest.mark.gpu


def cut(reader):
    sc = perturbed_scene(2, 0.4, 5)  # 64,000 particles: 4.6 MB of stresses
    parts, grid = scenes.setup_cut(sc)
    api.global_time_current = sc.params.dt
    lf = api.leap_frog(sc.n, grid.num_cell())
    stop, failed = threading.Event(), []

    def read():
        try:
            while not stop.is_set():
                for f in (_lib.F_S, _lib.F_POS, _lib.F_ID):
                    parts.download(f)
        except Exception as e:  # handed to the test's thread
            failed.append(e)

    t = threading.Thread(target=read)
    if reader:
        t.start()
    scenes.run(lf, parts, grid, 60)
    api.synchronize()
    stop.set()
    if reader:
        t.join()
    assert not failed, failed
    return {f: parts.download(f) for f in (_lib.F_ID, _lib.F_POS, _lib.F_VEL, _lib.F_RHO, _lib.F_S, _lib.F_T)}


def test_reads_do_not_disturb_steps(hip_device):
    alone, read = cut(False), cut(True)
    for f, a in alone.items():
        np.testing.assert_array_equal(a, read[f], err_msg=f"field {f}")
