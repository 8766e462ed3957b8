"""More plain systems than the GPU has CUs: every block size reaches the
states of a run of one system alone."""
import numpy as np
import pytest

from conftest import golden_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 128, 256])
def test_many_systems_reach_the_states_of_one(require_gpu, block):
    from sdmd_amd.engine import GpuEngine, System

    s, _ = golden_system("ala10ext")
    hot = s.arrays.copy()
    for f in ("vx", "vy", "vz"):
        hot.arr[f][1:] *= 1.25
    both = [s, System(None, hot)]
    alone = GpuEngine(both, block=256, max_pops=600)
    alone.prepare()
    alone.run(600)
    ref = [alone.state(k).arr for k in range(2)]
    alone.close()
    eng = GpuEngine([both[k % 2] for k in range(301)], block=block, max_pops=600)
    eng.prepare()
    eng.run(250)
    eng.run(350)
    for k in (0, 1, 127, 255, 256, 257, 299, 300):
        assert eng.stats(k)["error"] == 0 and eng.stats(k)["pops"] == 600
        got = eng.state(k).arr
        for f in ("x", "y", "z", "vx", "vy", "vz", "ev_time", "ev_partner", "ev_type", "ev_sub", "celllist"):
            assert np.array_equal(got[f], ref[k % 2][f]), (k, f)
    eng.close()
