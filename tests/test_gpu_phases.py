"""Per-phase device times of the plain engine: every phase that the entry
point names is timed, and together they make up the run."""
import numpy as np
import pytest

from conftest import golden_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,block", [("mix4x20", 256), ("ala10ext", 64)])
def test_every_phase_is_timed(require_gpu, name, block):
    from sdmd_amd.engine import GpuEngine

    s, _ = golden_system(name)
    eng = GpuEngine([s], block=block, profile=True, max_pops=4000)
    eng.prepare()
    before = np.array(list(eng.phase_times(0).values()))
    eng.run(4000)
    ms, times = eng.last_kernel_ms(), eng.phase_times(0)
    eng.close()
    assert all(t > 0 for t in times.values()), times
    total = 1e3 * (sum(times.values()) - before.sum())
    assert 0.7 * ms < total <= 1.02 * ms, (total, ms)      # between them: the launch and the tables' load
